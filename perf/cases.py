"""The work a user of this framework has it do, as cases that can be timed.

Five kinds of call, each through the package's public entry points:

``flow``     a run with a body in prescribed motion, from one write of the
             fields to the next: per step the marker kinematics and
             ``fluid_tsch``, and the whole state at the end.  The example
             inputs write their fields every 0.2 time units, which is 60 to
             200 steps at the time steps these grids take.
``coupled``  the reference's staggered coupling with a spring-mounted
             cylinder: per step the body, the markers, ``fluid_tsch``, the
             loads, the forcing check and the step's diagnostics, all read
             by the host.
``strong``   the iterated coupling: every step saved, repeated with new
             marker kinematics and rolled back between sub-iterations.
``batch``    many small runs on uneven grids advanced together.
``train``/``predict``  the network that proposes the first iterate of the
             iterated coupling.

``exact`` restates the flow step in float64 torch: cyclic reduction for the
line solves, a dense eigen-decomposition along both axes for the pressure,
everything else from the scheme's formulas.
"""
import functools
import math

import numpy as np
import torch

from fribois2d_amd import cases as fc
from fribois2d_amd import coupling, gpu, predictor

LZ, LY = 40.0, 30.0                 # domain: flow direction z, channel direction y
BODY_Z = 10.0                       # the body's place along z


def listed():
    return [
        # the smallest run anyone makes (the size of the quick checks):
        # launches and latency, hardly any arithmetic
        {"name": "flow_64x48", "kind": "flow", "n3m": 64, "n2m": 48, "mirror": True, "order": "auto", "graph": False,
         "dt": 0.0, "steps": 20},
        # the everyday cylinder grid (D/40 in the core), symmetric about the
        # channel centre, replayed as a graph
        {"name": "flow_384x288_graph", "kind": "flow", "n3m": 384, "n2m": 288, "mirror": True, "order": "auto",
         "graph": True, "dt": 0.0, "steps": 60},
        # a channel with more points across than along it: the transform has
        # to run along z, the reference's own order
        {"name": "flow_480x600_tall", "kind": "flow", "n3m": 480, "n2m": 600, "mirror": True, "order": "z",
         "graph": False, "dt": 0.0, "steps": 60},
        # the size, the fixed time step and the unsymmetric stretching of the
        # oscillating-cylinder example
        {"name": "flow_810x672_fixed_dt", "kind": "flow", "n3m": 810, "n2m": 672, "mirror": False, "order": "auto",
         "graph": False, "dt": 1.0e-3, "steps": 100},
        # odd counts in both directions: nothing divides a tile or a chunk
        {"name": "flow_1301x977_odd", "kind": "flow", "n3m": 1301, "n2m": 977, "mirror": True, "order": "auto",
         "graph": False, "dt": 0.0, "steps": 60},
        # the largest: the grid of the headline benchmark
        {"name": "flow_2048x1536", "kind": "flow", "n3m": 2048, "n2m": 1536, "mirror": True, "order": "auto",
         "graph": False, "dt": 0.0, "steps": 60},
        # staggered coupling on the everyday grid, everything the driver
        # reads back each step
        {"name": "coupled_384x288", "kind": "coupled", "n3m": 384, "n2m": 288, "steps": 20},
        # iterated coupling at mass ratio one on the predictor's grid
        {"name": "strong_512x384", "kind": "strong", "n3m": 512, "n2m": 384, "steps": 4, "iters": 5},
        # a parameter sweep: uneven small grids, some symmetric and some not
        {"name": "batch_24", "kind": "batch", "members": 24, "lo": 96, "hi": 448, "steps": 20},
        # the predictor's training set, a few epochs of minibatches of 256
        {"name": "train_2048", "kind": "train", "ni": 45, "no": 3, "n": 2048, "batch": 256, "epochs": 4},
        # one proposal, as the coupling loop asks for it at every step
        {"name": "predict_1", "kind": "predict", "ni": 45, "no": 3, "n": 1},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["flow", "flow", "flow", "coupled", "strong", "batch", "train", "predict"])
    if kind == "flow":
        n3m = _log(rng, 48, 2000)
        n2m = max(40, int(n3m * rng.uniform(0.6, 1.2)))
        n2m = min(n2m, 1500)
        tall = n2m >= n3m
        if tall:                     # the z order costs more per cell: stay below the largest listed run
            n3m, n2m = min(n3m, 900), min(n2m, 1080)
        return {"kind": "flow", "n3m": n3m, "n2m": n2m, "mirror": rng.random() < 0.5,
                "order": "z" if tall or rng.random() < 0.15 and n3m < 900 else "auto", "graph": rng.random() < 0.5,
                "dt": rng.choice([0.0, 1.0e-3]), "steps": rng.randint(20, 50)}
    if kind == "coupled":
        n3m = _log(rng, 96, 900)
        return {"kind": "coupled", "n3m": n3m, "n2m": int(n3m * rng.uniform(0.65, 0.95)), "steps": rng.randint(8, 24)}
    if kind == "strong":
        n3m = _log(rng, 128, 640)
        return {"kind": "strong", "n3m": n3m, "n2m": int(n3m * rng.uniform(0.65, 0.9)), "steps": rng.randint(2, 4),
                "iters": rng.randint(3, 6)}
    if kind == "batch":
        lo = rng.randint(64, 160)
        return {"kind": "batch", "members": rng.randint(4, 28), "lo": lo, "hi": lo + rng.randint(64, 280),
                "steps": rng.randint(8, 20)}
    if kind == "train":
        return {"kind": "train", "ni": rng.randint(9, 120), "no": rng.randint(1, 6), "n": _log(rng, 200, 6000),
                "batch": rng.choice([64, 100, 128, 256, 500]), "epochs": rng.randint(1, 4)}
    return {"kind": "predict", "ni": rng.randint(9, 120), "no": rng.randint(1, 6), "n": _log(rng, 1, 4000)}


# --------------------------------------------------------------------------
# grids and bodies

def _grid(n3m, n2m, mirror):
    """Node coordinates (rc, zz) and the body's y: a uniform core around the
    body and cubic stretching outside it, symmetric about the channel centre
    (mirror) or with the core below it."""
    n3, n2 = n3m + 1, n2m + 1
    zc = int(round(0.6 * n3))
    zb = max(3, int(round(0.12 * n3)))
    zz = fc.cubicstr([8.0, 16.0], [zb, zc, n3 - zb - zc], 0.0, LZ)
    yc = int(round(0.5 * n2))
    yc -= (n2 - yc) % 2
    body_y = 0.5 * LY if mirror else 0.4 * LY
    yb = (n2 - yc) // 2
    rc = fc.cubicstr([body_y - 2.0, body_y + 2.0], [yb, yc, n2 - yb - yc], 0.0, LY)
    return rc, zz, body_y


def _params(rc, zz, dt):
    re = 100.0
    return fc.FluidParams(n2=rc.size, n3=zz.size, alx3=LZ, rext2=LY, visc=1.0 / re, idtv=dt > 0.0, dt0=dt or 1.0e-3)


@functools.lru_cache(maxsize=16)
def _decomposition(n3m, n2m, mirror):
    """The phini inputs of a grid, which a program computes once and keeps."""
    rc, zz, _ = _grid(n3m, n2m, mirror)
    return fc.phini(zz, LZ)


class _Body:
    """A cylinder of diameter one heaving by 0.1 at frequency 0.2: rest
    positions once, kinematics at time t per step."""

    def __init__(self, zz, body_y, seed):
        core = np.diff(zz).min()
        nlm = int(min(1000, max(63, round(math.pi / core))))
        th = np.linspace(0.0, 2.0 * math.pi, nlm + 1)
        v = np.stack([0.5 * np.sin(th) + body_y, 0.5 * np.cos(th) + BODY_Z], axis=1)
        self.mid, self.lmA = 0.5 * (v[:-1] + v[1:]), np.hypot(*(v[1:] - v[:-1]).T)
        self.w = 2.0 * math.pi * 0.2
        self.phase = 2.0 * math.pi * np.random.default_rng(seed).random()
        self.cc = np.asfortranarray(self.mid)
        self.vel = np.zeros_like(self.cc, order="F")

    def at(self, t):
        a = self.w * t + self.phase
        np.add(self.mid[:, 0], 0.1 * (math.sin(a) - math.sin(self.phase)), out=self.cc[:, 0])
        self.vel[:, 0] = 0.1 * self.w * math.cos(a)
        return self.cc, self.vel, self.lmA


def _state(p, rc, zz, body_y, seed):
    """A run under way: the impulsive start with its seeded perturbation, plus
    a street of vortices from the body to the outflow, from a stream function
    at the cell corners (so its divergence vanishes cell by cell)."""
    st = fc.initial_state(p, seed)
    n2m, n3m = p.n2 - 1, p.n3 - 1
    phase = 2.0 * math.pi * np.random.default_rng([seed, 1]).random()
    ramp = np.clip((zz - BODY_Z) / 4.0, 0.0, 1.0)
    ramp = ramp * ramp * (3.0 - 2.0 * ramp)
    psi = 0.12 * np.outer(np.exp(-((rc - body_y) / 1.5) ** 2), ramp * np.sin(2.0 * math.pi * zz / 4.3 + phase))
    v = -np.diff(psi, axis=1) / np.diff(zz)[None, :]
    w = np.diff(psi, axis=0) / np.diff(rc)[:, None]
    v[0] = v[-1] = 0.0
    st["q2"][:, 3:n3m + 3] += v
    st["q3"][:n2m, 3:n3m + 4] += w
    st["qb2n"][:] += v[:, -1]
    st["qb3n"][:n2m] += w[:, -1]
    return st


def _members(case):
    """Sizes of a sweep's members: part of the case, not of its inputs."""
    rng = np.random.default_rng([case["members"], case["lo"], case["hi"]])
    out = []
    for _ in range(case["members"]):
        n3m = int(rng.integers(case["lo"], case["hi"] + 1))
        out.append((n3m, int(n3m * rng.uniform(0.65, 0.85)), bool(rng.integers(2))))
    return out


def _flow_instance(n3m, n2m, mirror, dt, seed):
    rc, zz, body_y = _grid(n3m, n2m, mirror)
    p = _params(rc, zz, dt)
    return p, rc, zz, _state(p, rc, zz, body_y, seed), _Body(zz, body_y, seed)


def _mlp_data(case, seed):
    """Inputs of unit spread as the predictor scales them, targets that depend
    on them, Glorot-uniform parameters."""
    rng = np.random.default_rng([seed, 3])
    ni, no, n, h = case["ni"], case["no"], case["n"], 64
    X = rng.standard_normal((n, ni)).astype(np.float32)
    T = (np.tanh(X @ (rng.standard_normal((ni, no)) / math.sqrt(ni))) + 0.05 * rng.standard_normal((n, no)))
    parts = []
    for rows, cols in ((h, ni), (h, h), (no, h)):
        parts += [rng.uniform(-1, 1, rows * cols) * math.sqrt(6.0 / (rows + cols)), 0.01 * rng.standard_normal(rows)]
    return X, T.astype(np.float32), np.concatenate(parts).astype(np.float32)


# --------------------------------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    if kind == "flow":
        p, rc, zz, st, body = _flow_instance(case["n3m"], case["n2m"], case["mirror"], case["dt"], seed)
        g = gpu.FluidStep(p, rc, zz, *_decomposition(case["n3m"], case["n2m"], case["mirror"]))
        g.set_transform(case["order"])
        g.set_graph(case["graph"])
        g.set_state(st)
        return {"kind": kind, "g": g, "body": body, "t": 0.0, "dt": p.dt0, "ns": 0, "steps": case["steps"]}
    if kind == "coupled":
        rc, zz, body_y = _grid(case["n3m"], case["n2m"], True)
        p = _params(rc, zz, 2.0e-3)
        g = gpu.FluidStep(p, rc, zz, *_decomposition(case["n3m"], case["n2m"], True))
        g.set_state(_state(p, rc, zz, body_y, seed))
        nlm = int(min(1000, max(63, round(math.pi / np.diff(zz).min()))))
        v0 = 0.05 + 0.1 * np.random.default_rng(seed).random()
        body = coupling.RigidBody(vert=fc.cylinder_vertices(body_y, BODY_Z, 0.5, nlm), cm=(body_y, BODY_Z, 0.0),
                                  rbden=10.0, rba=(0.78539816, 0.09817477), kk=(12.25, 0.0, 0.0), rbmcon=(0, 1, 1),
                                  cmv=np.array([v0, 0.0, 0.0]))
        return {"kind": kind, "g": g, "body": body, "loads": (np.zeros(2), 0.0), "dt": p.dt0, "ns": 0,
                "steps": case["steps"]}
    if kind == "strong":
        c, p, body = predictor.coupled_case(seed, case["n3m"], case["n2m"])
        g = gpu.FluidStep(p, c.rc, c.zz)
        g.set_state(_state(p, c.rc, c.zz, c.center[0], seed))
        return {"kind": kind, "g": g, "body": body, "loads": (np.zeros(2), 0.0), "dt": p.dt0, "ns": 0,
                "steps": case["steps"], "iters": case["iters"], "aitken": {}}
    if kind == "batch":
        gs, bodies, dts = [], [], []
        for i, (n3m, n2m, mirror) in enumerate(_members(case)):
            p, rc, zz, st, body = _flow_instance(n3m, n2m, mirror, 0.0, seed * 64 + i)
            g = gpu.FluidStep(p, rc, zz, *_decomposition(n3m, n2m, mirror))
            g.set_state(st)
            g.set_markers(*body.at(0.0))
            gs.append(g)
            bodies.append(body)
            dts.append(p.dt0)
        return {"kind": kind, "gs": gs, "b": gpu.FluidBatch(gs), "bodies": bodies, "t": np.zeros(len(gs)),
                "dt": np.array(dts), "ns": 0, "steps": case["steps"]}
    X, T, p0 = _mlp_data(case, seed)
    net = gpu.Mlp(case["ni"], case["no"], params=p0)
    return {"kind": kind, "net": net, "X": X, "T": T, "batch": case.get("batch"), "epochs": case.get("epochs")}


def run(state):
    return {"flow": _run_flow, "coupled": _run_coupled, "strong": _run_strong, "batch": _run_batch,
            "train": _run_train, "predict": _run_predict}[state["kind"]](state)


def _run_flow(s):
    g, body = s["g"], s["body"]
    t, dt, ns = s["t"], s["dt"], s["ns"]
    dts = np.empty(s["steps"])
    for i in range(s["steps"]):
        g.set_markers(*body.at(t))
        dt, _ = g.fluid_tsch(ns, dt, dt)
        t += dt
        ns += 1
        dts[i] = dt
    s["t"], s["dt"], s["ns"] = t, dt, ns
    return {"dt": dts, "state": g.get_state()}


def _run_coupled(s):
    g, body = s["g"], s["body"]
    hist = []
    for _ in range(s["steps"]):
        s["loads"], _, cflm = coupling.weak_step(g, body, s["loads"], s["ns"], s["dt"])
        _, _, nv, nw = g.checkbcs()
        d = g.diagnostics()
        f, m = s["loads"]
        hist.append((body.cm[0], body.cmv[0], f[0], f[1], m, cflm, nv, nw, d["ektot"], d["vmax2"], d["vmax3"]))
        s["ns"] += 1
    return {"hist": np.array(hist), "state": g.get_state()}


def _run_strong(s):
    g = s["g"]
    hist = []
    for _ in range(s["steps"]):
        s["loads"], s["body"], _, _, _ = coupling.strong_step(g, s["body"], s["loads"], s["ns"], s["dt"], tol=0.0,
                                                              maxit=s["iters"], state=s["aitken"], strict=False)
        f, m = s["loads"]
        hist.append((s["body"].cm[0], s["body"].cmv[0], f[0], f[1], m))
        s["ns"] += 1
    return {"hist": np.array(hist), "state": g.get_state()}


def _run_batch(s):
    b, t, dt = s["b"], s["t"], s["dt"]
    for _ in range(s["steps"]):
        b.set_markers([body.at(ti) for body, ti in zip(s["bodies"], t)])
        dt, _, err = b.step(s["ns"], dt, dt)
        if err.any():
            raise RuntimeError(f"instance errors {err}")
        t = t + dt
        s["ns"] += 1
    s["t"], s["dt"] = t, dt
    fields = [g.get_state() for g in s["gs"]]
    return {"dt": dt, **{k: np.concatenate([f[k].ravel(order="F") for f in fields]) for k in fields[0]}}


def _run_train(s):
    loss = s["net"].train(s["X"], s["T"], s["epochs"], s["batch"], 2e-3)
    return {"loss": np.float32(loss), "params": s["net"].params()}


def _run_predict(s):
    return s["net"].predict(s["X"])


# --------------------------------------------------------------------------
# what a pass cannot do without

def _step_work(n3m, n2m, mirror, order):
    """Bytes and flops of one time step.  Per substep every field that the
    scheme's stages must read or write once per sweep over the grid (the
    right-hand sides 9, the two line sweeps 4 and 6, the divergence 3, the
    transforms and mode lines 6, the projection 7), plus the transform
    matrices; the flops of the transforms (2 n^2 per line point and
    direction, half that on a symmetric grid) and about 300 per cell."""
    cells = n3m * n2m
    along_y = order == "auto" and n2m < n3m
    n = n2m if along_y else n3m
    half = 0.5 if along_y and mirror and n2m % 2 == 0 else 1.0
    return {"bytes": 3 * (35 * 8 * cells + 16 * n * n * half) + 16 * cells, "flops": 3 * (4 * cells * n * half + 300 * cells)}


def work(case):
    kind = case["kind"]
    if kind in ("flow", "coupled", "strong"):
        w = _step_work(case["n3m"], case["n2m"], case.get("mirror", True), case.get("order", "auto"))
        reps = case["steps"] * case.get("iters", 1)
        out = 40 * case["n3m"] * case["n2m"]
        return {"bytes": reps * w["bytes"] + 2 * out, "flops": reps * w["flops"]}
    if kind == "batch":
        ws = [_step_work(a, b, m, "auto") for a, b, m in _members(case)]
        out = sum(80 * a * b for a, b, _ in _members(case))
        return {"bytes": case["steps"] * sum(w["bytes"] for w in ws) + out, "flops": case["steps"] * sum(w["flops"] for w in ws)}
    ni, no, n = case["ni"], case["no"], case["n"]
    np_ = 64 * ni + 64 + 64 * 64 + 64 + no * 64 + no
    mac = 64 * ni + 64 * 64 + no * 64
    if kind == "train":
        steps = case["epochs"] * -(-n // case["batch"])
        return {"bytes": case["epochs"] * 4 * n * (ni + no) + steps * 24 * np_, "flops": case["epochs"] * n * 6.0 * mac}
    return {"bytes": 4 * (np_ + n * (ni + no)), "flops": 2.0 * n * mac}


# --------------------------------------------------------------------------
# float64 values without this package's step

def exact(case, seed):
    kind = case["kind"]
    if kind == "flow":
        inst = _flow_instance(case["n3m"], case["n2m"], case["mirror"], case["dt"], seed)
        dts, state = _exact_flow(*inst, case["steps"])
        return {"dt": dts, "state": state}
    if kind == "batch":
        ends, states = [], []
        for i, (n3m, n2m, mirror) in enumerate(_members(case)):
            dts, state = _exact_flow(*_flow_instance(n3m, n2m, mirror, 0.0, seed * 64 + i), case["steps"])
            ends.append(dts[-1])
            states.append(state)
        return {"dt": np.array(ends), **{k: np.concatenate([s[k].ravel(order="F") for s in states]) for k in states[0]}}
    if kind == "train":
        return _exact_train(case, seed)
    if kind == "predict":
        X, _, p0 = _mlp_data(case, seed)
        return _mlp_forward(_mlp_split(torch.from_numpy(p0).double(), case), torch.from_numpy(X).double())[2].numpy()
    return None     # coupled runs: their flow is the flow cases', their loads have no value of another origin


def _mlp_split(p, case):
    ni, no, h, at, out = case["ni"], case["no"], 64, 0, []
    for shape in ((h, ni), (h,), (h, h), (h,), (no, h), (no,)):
        k = math.prod(shape)
        out.append(p[at:at + k].reshape(shape))
        at += k
    return out


def _mlp_forward(w, x):
    h1 = torch.tanh(x @ w[0].T + w[1])
    h2 = torch.tanh(h1 @ w[2].T + w[3])
    return h1, h2, h2 @ w[4].T + w[5]


def _exact_train(case, seed):
    X, T, p0 = _mlp_data(case, seed)
    X, T, p = torch.from_numpy(X).double(), torch.from_numpy(T).double(), torch.from_numpy(p0).double()
    m, v, step, loss, lr = torch.zeros_like(p), torch.zeros_like(p), 0, 0.0, float(np.float32(2e-3))
    for _ in range(case["epochs"]):
        for at in range(0, case["n"], case["batch"]):
            x, t = X[at:at + case["batch"]], T[at:at + case["batch"]]
            q = p.clone().requires_grad_(True)
            y = _mlp_forward(_mlp_split(q, case), x)[2]
            loss = ((y - t) ** 2).mean()
            loss.backward()
            step += 1
            m = 0.9 * m + 0.1 * q.grad
            v = 0.999 * v + 0.001 * q.grad ** 2
            p = p - lr * (m / (1 - 0.9 ** step)) / ((v / (1 - 0.999 ** step)).sqrt() + 1e-8)
    return {"loss": float(loss), "params": p.numpy()}


class _Eig:
    """Eigen-decomposition of a tridiagonal operator (rows lo, di, up) that a
    diagonal scaling makes symmetric."""

    def __init__(self, lo, di, up, dev):
        s = np.concatenate([[0.0], np.cumsum(0.5 * np.log(lo[1:] / up[:-1]))])
        s = np.exp(s - s.mean())
        off = np.sqrt(lo[1:] * up[:-1])
        w, q = np.linalg.eigh(np.diag(di) + np.diag(off, 1) + np.diag(off, -1))
        self.w = torch.from_numpy(w).to(dev)
        self.V = torch.from_numpy(s[:, None] * q).to(dev)
        self.Vi = torch.from_numpy(np.ascontiguousarray(q.T / s[None, :])).to(dev)


def _line_solve(op, bd, r, dim):
    """(1 - bd L) x = r along dimension `dim` of r, L tridiagonal (rows lo,
    di, up), by cyclic reduction of all rows at once."""
    n = r.shape[dim]
    lo, di, up = (-bd * op[0], 1.0 - bd * op[1], -bd * op[2])
    lo, up = lo.clone(), up.clone()
    lo[0] = up[-1] = 0.0

    def shift(x, h, d, fill):
        pad = x.narrow(d, 0, abs(h)) * 0.0 + fill
        return torch.cat([pad, x.narrow(d, 0, x.shape[d] - h)], d) if h > 0 else torch.cat([x.narrow(d, -h, x.shape[d] + h), pad], d)

    h = 1
    while h < n:
        a, c = lo / shift(di, h, 0, 1.0), up / shift(di, -h, 0, 1.0)
        a2, c2 = (a, c) if dim == 1 else (a[:, None], c[:, None])
        r = r - a2 * shift(r, h, dim, 0.0) - c2 * shift(r, -h, dim, 0.0)
        di = di - a * shift(up, h, 0, 0.0) - c * shift(lo, -h, 0, 0.0)
        lo, up = -a * shift(lo, h, 0, 0.0), -c * shift(up, -h, 0, 0.0)
        h *= 2
    return r / (di if dim == 1 else di[:, None])


def _exact_flow(p, rc, zz, st, body, steps):
    """`steps` time steps of the scheme (three Runge-Kutta substeps, free-slip
    walls, moving-least-squares forcing) on arrays [k, j], in float64."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    n2, n3 = p.n2, p.n3
    n2m, n3m = n2 - 1, n3 - 1

    def T(a):
        return torch.from_numpy(np.ascontiguousarray(a)).to(dev)

    # metrics: cell widths, distances of cell centres (whole cells at the ends)
    hy, hz = np.diff(rc), np.diff(zz)

    def centre(h):
        c = np.empty(h.size + 1)
        c[0], c[-1] = h[0], h[-1]
        c[1:-1] = 0.5 * (h[1:] + h[:-1])
        return c

    cy, cz = centre(hy), centre(hz)
    iy, iz, icy, icz = T(1.0 / hy), T(1.0 / hz), T(1.0 / cy), T(1.0 / cz)
    # second differences: at interior nodes (q2 along y, q3 along z) and at
    # cell centres (q3 along y: no flux through the walls; q2 along z: Dirichlet
    # half a cell outside, which counts a whole cell twice; pressure: no flux)
    node = {}
    for d, h, c in (("y", hy, cy), ("z", hz, cz)):
        lo, up = 1.0 / (c[1:-1] * h[:-1]), 1.0 / (c[1:-1] * h[1:])
        node[d] = (lo, -(lo + up), up)
    cen = {}
    for d, h, c in (("y", hy, cy), ("z", hz, cz)):
        lo, up = 1.0 / (h * c[:-1]), 1.0 / (h * c[1:])
        l0, u0 = lo.copy(), up.copy()
        l0[0] = u0[-1] = 0.0
        cen[d] = (l0, -(l0 + u0), u0, lo, up)
    sk = (cen["z"][0], cen["z"][1].copy(), cen["z"][2])
    sk[1][0] -= 2.0 * cen["z"][3][0]
    sk[1][-1] -= 2.0 * cen["z"][4][-1]
    k_in, k_out = 2.0 * cen["z"][3][0], 2.0 * cen["z"][4][-1]
    Ey, Ez = _Eig(*cen["y"][:3], dev), _Eig(*cen["z"][:3], dev)
    L2j, L3j, L2k = (tuple(T(a) for a in op) for op in (node["y"], cen["y"][:3], sk))
    L3k = tuple(a[1:] for a in L2k)
    k3_last = float(sk[2][-1]) if sk[2][-1] else 0.0     # coupling of q3's last row to the outflow plane
    wn2 = tuple(T(a) for a in node["y"])
    wc3 = tuple(T(a) for a in cen["y"][:3])
    wnz = tuple(T(a)[:, None] for a in node["z"])
    wsk = tuple(T(a)[:, None] for a in sk)

    def field(a):
        return T(a.T).clone()

    q2, q3, pr = (field(st[f]) for f in ("q2", "q3", "pr"))          # [k + 2, j - 1]
    ru2, ru3 = field(st["ru2"]), field(st["ru3"])
    bc = {k: T(st[k]).clone() for k in ("qb2s", "qb3s", "qb2n", "qb3n", "dq2x2o", "dq3x2o")}
    K = slice(3, n3m + 3)                                            # planes 1..n3m
    J = slice(0, n2m)                                                # columns 1..n2m
    dy, dz = T(hy), T(hz)
    re = 1.0 / p.visc
    ga_, ro_ = (8 / 15, 5 / 12, 3 / 4), (0.0, -17 / 60, -5 / 12)
    rm, zm = 0.5 * (rc[1:] + rc[:-1]), 0.5 * (zz[1:] + zz[:-1])
    ynode, znode = (rc, np.append(rm, rc[-1])), (np.append(zm, zz[-1]), zz)

    def pad_end(x):
        return np.append(x, x[-1])

    def support(pos, lmA):
        """Cells, weights and volume factors of every marker, both components."""
        out = []
        for d in (0, 1):
            y, z = ynode[d], znode[d]
            n = pos.shape[0]
            j0 = np.abs(y[None, :] - pos[:, :1]).argmin(1)
            k0 = np.abs(z[None, :] - pos[:, 1:]).argmin(1)
            jj = (j0[:, None] + np.array([-1, -1, -1, 0, 0, 0, 1, 1, 1])[None, :])
            kk = (k0[:, None] + np.array([-1, 0, 1] * 3)[None, :])
            yp, zp = pad_end(y), pad_end(z)
            sy, sz, ey, ez = yp[jj], zp[kk], yp[jj + 1] - yp[jj], zp[kk + 1] - zp[kk]

            def w1(r):
                a = 2 / 3 - 4 * r ** 2 + 4 * r ** 3
                b = 4 / 3 - 4 * r + 4 * r ** 2 - 4 / 3 * r ** 3
                return np.where(r > 1.0, 0.0, np.where(r <= 0.5, a, b))

            w = w1(np.abs(pos[:, :1] - sy) / (p.radiusSD * ey)) * w1(np.abs(pos[:, 1:] - sz) / (p.radiusSD * ez))
            # the basis about the marker: the same fit, better conditioned
            P = np.stack([np.ones_like(sy), sy - pos[:, :1], sz - pos[:, 1:]], axis=1)
            A = np.einsum("nm,nam,nbm->nab", w, P, P)
            e1 = np.zeros((n, 3, 1))
            e1[:, 0] = 1.0
            phi = (np.linalg.solve(A, e1)[:, :, 0][:, :, None] * P).sum(1) * w
            cl = lmA * (0.5 * phi * (ey + ez)).sum(1) / (phi * ey * ez).sum(1)
            out.append((T(jj), T(kk), T(phi), T(cl)))
        return out

    t, dt, dts = 0.0, p.dt0, []
    for ns in range(steps):
        cc, vel, lmA = body.at(t)
        mk, vel = support(np.array(cc), lmA), T(np.array(vel))
        if not p.idtv and ns > 0:
            c = ((q2[K, :n2m] + q2[K, 1:n2]) * 0.5 * iy).abs() + ((q3[K, J] + q3[4:n3m + 4, J]) * 0.5 * iz[:, None]).abs()
            dt = min(p.cflmax / max(float(c.max()), 1e-8), p.dtmax)
        dts.append(dt)
        t += dt
        beta = 0.5 * dt / re
        for ga, ro in zip(ga_, ro_):
            al = ga + ro
            bd = beta * al
            # convective outflow, corrected to the inflow's flux
            d2 = (bc["qb2n"][J] - q2[n3m + 2, J]) * 2.0 * icz[-1]
            d3 = (bc["qb3n"][J] - q3[n3m + 2, J]) * icz[-1]
            dqb2n = -dt * (ga * d2 + ro * bc["dq2x2o"][J]) * p.cou
            dqb3n = -dt * (ga * d3 + ro * bc["dq3x2o"][J]) * p.cou
            bc["dq2x2o"][J], bc["dq3x2o"][J] = d2, d3
            dqb3n = dqb3n - (dqb3n * dy).sum() / dy.sum()
            # right-hand sides
            a2, b2 = q2[K, :n2m], q2[K, 1:n2]
            a3 = q3[3:n3m + 4, J]                                    # planes 1..n3
            P = pr[K, J]
            fyy = ((a2 + b2) ** 2) * 0.25                            # q2 q2 at cell centres
            c2 = (fyy[:, 1:] - fyy[:, :-1]) * icy[1:-1]
            q3c = a3[:, 1:] + a3[:, :-1]                             # twice q3 at q2's columns, planes 1..n3
            z = q2[K, 1:n2m]
            corner = q3c[1:n3m] * (z[1:] + z[:-1]) * 0.25
            inflow = (bc["qb2s"][1:n2m] * (bc["qb3s"][1:n2m] + bc["qb3s"][:n2m - 1]) * 0.5)[None]
            outflow = (bc["qb2n"][1:n2m] * (bc["qb3n"][1:n2m] + bc["qb3n"][:n2m - 1]) * 0.5)[None]
            flux = torch.cat([inflow, corner, outflow])
            conv2 = -(c2 + (flux[1:] - flux[:-1]) * iz[:, None])
            yy = q2[K, 2:n2] * wn2[2] + z * wn2[1] + q2[K, 0:n2m - 1] * wn2[0]
            zm_, zp_ = torch.cat([z[:1] * 0, z[:-1]]), torch.cat([z[1:], z[:1] * 0])
            zz2 = zp_ * wsk[2] + z * wsk[1] + zm_ * wsk[0]
            zz2[0] += bc["qb2s"][1:n2m] * k_in
            zz2[-1] += bc["qb2n"][1:n2m] * k_out
            grad2 = al * icy[1:-1] * (P[:, 1:] - P[:, :-1])
            r2 = (ga * conv2 + ro * ru2[:, 1:n2m] + al / re * (yy + zz2) - grad2) * dt
            ru2[:, 1:n2m] = conv2
            m3 = a3[1:n3m]                                           # q3, planes 2..n3m
            w2 = q2[4:n3m + 3, 0:n2] + q2[3:n3m + 2, 0:n2]           # twice q2 at q3's planes
            side = torch.cat([2.0 * m3[:, :1], m3[:, 1:] + m3[:, :-1], 2.0 * m3[:, -1:]], dim=1)
            f32 = w2 * side * 0.25
            fzz = (q3[3:n3m + 3, J] + q3[4:n3m + 4, J]) ** 2 * 0.25
            conv3 = -((f32[:, 1:] - f32[:, :-1]) * iy + (fzz[1:] - fzz[:-1]) * icz[1:-1, None])
            conv3[-1] = 0.0                                          # the scheme leaves the last plane's at zero
            e = torch.cat([m3[:, 1:], m3[:, :1] * 0], dim=1)
            w = torch.cat([m3[:, :1] * 0, m3[:, :-1]], dim=1)
            y3 = e * wc3[2] + m3 * wc3[1] + w * wc3[0]
            z3 = q3[5:n3m + 4, J] * wnz[2] + m3 * wnz[1] + q3[3:n3m + 2, J] * wnz[0]
            r3 = (ga * conv3 + ro * ru3[1:, J] + al / re * (y3 + z3) - al * icz[1:-1, None] * (P[1:] - P[:-1])) * dt
            ru3[1:, J] = conv3
            # forcing at the markers
            R2 = torch.zeros(n3m, n2, dtype=torch.float64, device=dev)
            R3 = torch.zeros_like(R2)
            R2[:, 1:n2m], R3[1:, J] = r2, r3
            if p.ibact:
                for R, q, (jj, kk, phi, cl), u in ((R2, q2, mk[0], vel[:, 0]), (R3, q3, mk[1], vel[:, 1])):
                    pred = q[K] + R
                    f = (u - (phi * pred[kk, jj]).sum(1)) * cl
                    add = torch.zeros_like(R)
                    add.index_put_((kk, jj), phi * f[:, None], accumulate=True)
                    add[-1] = 0.0
                    R += add
            r2, r3 = R2[:, 1:n2m], R3[1:, J]
            # (1 - bd Lyy)(1 - bd Lzz) dq = r, line by line along y, then z
            r2 = _line_solve(L2j, bd, r2, 1)
            r2[-1] += bd * k_out * dqb2n[1:]
            r2 = _line_solve(L2k, bd, r2, 0)
            r3 = _line_solve(L3j, bd, r3, 1)
            r3[-1] += bd * k3_last * dqb3n
            r3 = _line_solve(L3k, bd, r3, 0)
            q2[K, 1:n2m] += r2
            q3[4:n3m + 3, J] += r3
            q3[n3m + 3, J] += dqb3n
            # pressure increment; its free constant is fixed by a zero mean along
            # the last row (only the pressure outside the interior shows it)
            div = ((q2[K, 1:n2] - q2[K, :n2m]) * iy + (q3[4:n3m + 4, J] - q3[K, J]) * iz[:, None]) / (dt * al)
            h = Ez.Vi @ div @ Ey.Vi.T
            lam = Ez.w[:, None] + Ey.w[None, :]
            zero = lam.abs() == lam.abs().min()
            h = torch.where(zero, torch.zeros_like(h), h / lam)
            phi = Ez.V @ h @ Ey.V.T
            phi -= (dz * phi[:, -1]).sum() / dz.sum()
            q2[K, 1:n2m] -= (phi[:, 1:] - phi[:, :-1]) * (al * dt * icy[1:-1])
            q3[4:n3m + 3, J] -= (phi[1:] - phi[:-1]) * (al * dt * icz[1:-1, None])
            pr[K, J] += phi - bd * div
            pr -= (pr[K, J] * dz[:, None] * dy).sum() / (p.rext2 * p.alx3)
            bc["qb2n"][J] += dqb2n
            bc["qb3n"][J] += dqb3n
    state = {"q2": q2, "q3": q3, "pr": pr, "ru2": ru2, "ru3": ru3}
    state = {k: np.asfortranarray(v.cpu().numpy().T) for k, v in state.items()}
    state.update({k: v.cpu().numpy() for k, v in bc.items()})
    return np.array(dts), state
