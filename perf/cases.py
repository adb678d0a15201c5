"""Workloads of the IPC Newton step, each one call chain of a user's program.

Kinds:

* ``step``: a restart from a frame (positions and velocities) and a few whole
  time steps, returning the frame that follows;
* ``direction``: one Newton direction at the current positions -- constraint
  search, assembly, solve (the FP32 form solves loosely, then continues the
  solve of the direction that would decide the Newton test);
* ``linesearch``: the line search along a direction -- constraint search and
  energy at the start, step bound, collision test, constraint search and
  energy at the end;
* ``predict``: the learned warm start's increment at a step's start;
* ``mlp``: the warm-start network on host rows, forward or loss and gradient;
* ``ccd``: times of impact of host pairs.

Scenes: a ``slab`` of nx x ny x nz lattice vertices between two closing plates,
and a ``pile`` of layers x m x m cubes of n^3 vertices on a fixed ground.
"""
import ctypes
import functools
import math
import os

import numpy as np
import torch

from fastipc_amd import _lib
from fastipc_amd import scene as S
from fastipc_amd.newton import NewtonIPC
from fastipc_amd.warmstart import WEIGHTS_DIR, LearnedWarmStart, WarmStartMLP, scale_for

DENSITY, PILE_E, PILE_NU = 1000.0, 1e5, 0.4
NET = (16, 256, 4, 3)  # inputs, width, hidden layers, outputs of the warm-start network


def listed():
    """The smallest scene of the repository's configurations, its largest, and
    odd sizes between; both precisions; each layer of a step by itself."""
    return [
        # whole steps of a small slab in FP64: every launch is short, a pass
        # is latency (steps are taken of slabs only: the 200 to 400 solver
        # iterations of a stiff pile amplify a last bit into the frame, so
        # piles are measured by their directions and line searches)
        {"name": "step-slab-small", "kind": "step", "scene": "slab", "nx": 10, "ny": 16, "nz": 10,
         "fp32": False, "warm": False, "steps": 3},
        # the 1M-tet compressed slab of the benchmark, in its fastest form
        {"name": "step-slab-1m", "kind": "step", "scene": "slab", "nx": 50, "ny": 80, "nz": 50,
         "fp32": True, "warm": True, "steps": 4},
        # a Newton direction of two stacked cubes, the first configuration
        {"name": "direction-two-cubes", "kind": "direction", "scene": "pile", "n": 10, "m": 1, "layers": 2,
         "fp32": False},
        # an ordinary model of a ragged size
        {"name": "direction-slab-ragged", "kind": "direction", "scene": "slab", "nx": 23, "ny": 37, "nz": 29,
         "fp32": True},
        # the 27 cubes of the second configuration, stacked into contact
        {"name": "direction-27-cubes", "kind": "direction", "scene": "pile", "n": 16, "m": 3, "layers": 3,
         "fp32": False},
        {"name": "direction-slab-1m", "kind": "direction", "scene": "slab", "nx": 50, "ny": 80, "nz": 50,
         "fp32": True},
        {"name": "linesearch-two-cubes", "kind": "linesearch", "scene": "pile", "n": 10, "m": 1, "layers": 2},
        # the 200 small cubes of the third configuration: mostly surface, the
        # broad phase and the contact rows carry the pass
        {"name": "linesearch-200-cubes", "kind": "linesearch", "scene": "pile", "n": 8, "m": 5, "layers": 8},
        {"name": "linesearch-slab-1m", "kind": "linesearch", "scene": "slab", "nx": 50, "ny": 80, "nz": 50},
        # the warm start of a step of the benchmark: features and inference
        {"name": "predict-slab-1m", "kind": "predict", "scene": "slab", "nx": 50, "ny": 80, "nz": 50},
        # a training step of the warm-start network at its default batch
        {"name": "mlp-grad-8192", "kind": "mlp", "rows": 8192, "backward": True},
        # a caller with its own broad phase: edge pairs in host arrays
        {"name": "ccd-edges-30011", "kind": "ccd", "pairs": 30011, "edges": True},
    ]


def draw(rng):
    """Another case of the same ranges: 500 to 200,000 vertices, 64 to 200,000
    network rows, 16 to 100,000 pairs, sizes spread over their logarithm."""
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["step", "direction", "direction", "linesearch", "linesearch", "predict", "mlp", "ccd"])
    if kind == "mlp":
        backward = rng.random() < 0.6
        return {"kind": kind, "rows": log_int(64, 65536 if backward else 200000), "backward": backward}
    if kind == "ccd":
        return {"kind": kind, "pairs": log_int(16, 100000), "edges": rng.random() < 0.5}
    case = {"kind": kind}
    if kind in ("step", "predict") or rng.random() < 0.5:
        v = log_int(500, 200000)
        a, b = rng.uniform(0.6, 1.6), rng.uniform(0.6, 1.6)
        nx = max(4, int((v / (a * b)) ** (1 / 3)))
        ny, nz = max(4, int(nx * a)), max(4, int(nx * b))
        while nx * ny * nz > 200000:
            nz -= 1
        case |= {"scene": "slab", "nx": nx, "ny": ny, "nz": nz}
    else:
        m, layers = rng.randint(1, 5), rng.randint(1, 8)
        v = log_int(500, 110000)
        case |= {"scene": "pile", "n": min(20, max(3, int((v / (m * m * layers)) ** (1 / 3)))), "m": m,
                 "layers": layers}
    if kind in ("step", "direction"):
        case["fp32"] = rng.random() < 0.5
    if kind == "step":
        case |= {"warm": case["fp32"], "steps": rng.randint(1, 3)}
    return case


# ---- scenes and states ------------------------------------------------------
@functools.lru_cache(maxsize=4)
def _pile(n, m, layers):
    """layers x m x m cubes over a fixed ground, apart by 0.05 of their edge;
    odd layers are shifted so that no two edges of a stack are aligned."""
    xc, tc = S.lattice(n)
    edge = (n - 1) * S.LATTICE_SPACING
    gap = 0.05 * edge
    xs, ts, nv = [], [], 0
    for layer in range(layers):
        shift = (0.31 * edge, 0.17 * edge) if layer % 2 else (0.0, 0.0)
        for i in range(m):
            for k in range(m):
                xs.append(xc + [i * (edge + gap) + shift[0], gap + layer * (edge + gap), k * (edge + gap) + shift[1]])
                ts.append(tc + nv)
                nv += len(xc)
    width = m * (edge + gap)
    gx, gt = S.box([-edge, -0.1 * edge, -edge], [width + edge, 0.0, width + edge])
    ts.append(gt + nv)
    x, tets = np.concatenate(xs + [gx]), np.concatenate(ts).astype(np.int32)
    fixed = np.arange(len(x)) >= nv
    one = np.ones(len(tets))
    return S.Scene(name=f"pile_{layers}x{m}x{m}x{n}", x=x, tets=tets, density=DENSITY * one, youngs=PILE_E * one,
                   poisson=PILE_NU * one, dirichlet_mask=fixed, dt=0.01)


@functools.lru_cache(maxsize=2)
def _slab(nx, ny, nz):
    return S.compressed_slab(nx, ny, nz)


def _scene(case):
    if case["scene"] == "slab":
        return _slab(case["nx"], case["ny"], case["nz"])
    return _pile(case["n"], case["m"], case["layers"])


def _wave(rng, size, n=3):
    """A smooth field of zero mean and size about 1 over positions of extent size."""
    k = rng.uniform(0.5, 2.0, (n, 3)) * 2 * math.pi / size
    phase, amp = rng.uniform(0, 2 * math.pi, n), rng.uniform(-1, 1, (n, 3))
    return lambda x: sum(np.sin(x @ k[j] + phase[j])[:, None] * amp[j] for j in range(n)) / n


def _state(case, sc, seed):
    """Positions in contact without intersections, velocities, a search
    direction and the frame number, from the seed alone: the bodies are
    compressed by up to two percent, their facing surfaces lie 0.4 to 1.2
    barrier distances apart, and a smooth field and a little noise move
    everything."""
    rng = np.random.default_rng([seed, 77])
    x, free, dh = sc.x.copy(), ~sc.dirichlet_mask, sc.dhat
    strain = rng.uniform(0.002, 0.02)
    size = float(np.max(sc.x[free].max(0) - sc.x[free].min(0)))

    def gap(p, flip):
        """the gap to the surface below (above), over the horizontal plane"""
        a, b = rng.uniform(1.0, 3.0, 2) * 2 * math.pi / size
        return dh * (0.8 + 0.4 * np.sin(a * p[:, 0] + flip) * np.sin(b * p[:, 2] + flip))

    if case["scene"] == "slab":
        height = (case["ny"] - 1) * S.LATTICE_SPACING
        frame = int(math.ceil((0.004 * math.sqrt(sum(((case[k] - 1) * S.LATTICE_SPACING) ** 2 for k in
                                                     ("nx", "ny", "nz"))) + strain * height / 2) /
                              (0.1 * height * sc.dt)))
        plates = sc.dirichlet_rows((frame - 1) * sc.dt)[1]
        x[~free] = plates
        lo, hi = plates[:8, 1].max(), plates[8:, 1].min()
        p = sc.x[free]
        s = p[:, 1] / height
        bottom, top = lo + gap(p, 0.0), hi - gap(p, 1.0)
        x[free, 1] = bottom + s * (top - bottom)
        v = np.zeros_like(x)
        v[free, 1] = (0.5 - s) * 0.2 * height
        inside = s * (1 - s)
    else:
        n, frame = case["n"], 1
        edge = (n - 1) * S.LATTICE_SPACING
        layer = np.repeat(np.arange(case["layers"]), case["m"] ** 2 * n ** 3)
        p = sc.x[free]
        s = (p[:, 1] - (0.05 * edge + layer * 1.05 * edge)) / edge
        below = layer * edge * (1 - strain)
        g = gap(p, 0.0)
        x[free, 1] = below + g + s * (edge * (1 - strain) - g)
        v = np.zeros_like(x)
        v[free, 1] = -rng.uniform(0.02, 0.1)
        inside = s * (1 - s)
    field = _wave(rng, size)(sc.x[free]) * inside[:, None]
    x[free] += field * 0.1 * strain * size
    x[free] += rng.uniform(-0.02, 0.02, (int(free.sum()), 3)) * dh
    v[free] += _wave(rng, size)(sc.x[free]) * 0.02 * size
    # a direction of up to a few barrier distances, which closes some of the gaps
    d = np.zeros_like(x)
    d[free] = _wave(rng, size)(sc.x[free]) * rng.uniform(0.5, 3.0) * dh
    return x, v, d, frame


def _sim(case, seed):
    sc = _scene(case)
    x, v, d, frame = _state(case, sc, seed)
    sim = NewtonIPC(sc, precision=int(case.get("fp32", False)),
                    pcg_tol_search=2e-2 if case.get("fp32") else None, certify=bool(case.get("fp32")))
    # a step that ended at x with velocity v, then the start of the next one
    sim.set_state(x - sc.dt * v, v)
    sim.compute_xn_and_xTilde((frame - 1) * sc.dt)
    sim.set_vector(0, x)
    sim.compute_v()
    sim.compute_xn_and_xTilde(frame * sc.dt)
    sim.frame = frame
    sim.set_vector(1, d)
    sim.save_xPrev()
    return {"sim": sim, "scene": sc, "x": x, "v": v, "d": d, "frame": frame}


def _rows(case, seed):
    """Feature and target rows as the warm start sees them: increments of a
    fraction of the length scale, a few rows near a contact."""
    rng = np.random.default_rng([seed, 78])
    n = case["rows"]
    X = (0.3 * rng.standard_normal((n, NET[0]))).astype(np.float32)
    near = rng.random(n) < 0.1
    normal = rng.standard_normal((n, 3))
    normal /= np.linalg.norm(normal, axis=1)[:, None]
    X[:, 6], X[:, 7], X[:, 8] = 0.0, -0.02, 0.0
    X[:, 9] = np.where(near, rng.random(n), 1.0)
    X[:, 10:13] = np.where(near[:, None], normal, 0.0)
    X[:, 13] = 0.0
    X[:, 14:] = np.where(near[:, None], X[:, 14:], 0.0)
    return X, (0.05 * rng.standard_normal((n, NET[3]))).astype(np.float32)


@functools.lru_cache(maxsize=1)
def _weights():
    path = os.path.join(WEIGHTS_DIR, "ws_slab.npz")
    with np.load(path, allow_pickle=False) as d:
        return (d["bf16"].astype(np.uint32) << 16).view(np.float32)


def _pairs(case, seed):
    """Pairs of primitives of an edge length about 0.1, a few barrier
    distances apart, moving against each other by up to twice their distance."""
    rng = np.random.default_rng([seed, 79])
    n, e = case["pairs"], S.LATTICE_SPACING
    a = rng.uniform(-1, 1, (n, 3))
    along = rng.standard_normal((n, 2, 3))
    along *= e / np.linalg.norm(along, axis=2)[:, :, None]
    normal = np.cross(along[:, 0], along[:, 1])
    normal /= np.linalg.norm(normal, axis=1)[:, None]
    dist = rng.uniform(0.005, 0.05, n)
    b = a + normal * dist[:, None]
    if case["edges"]:  # two edges crossing at their middles
        p = [a - along[:, 0] / 2, a + along[:, 0] / 2, b - along[:, 1] / 2, b + along[:, 1] / 2]
        side = (1.0, 1.0, -1.0, -1.0)
    else:  # a point over a triangle
        c = b - (along[:, 0] + along[:, 1]) / 3
        p = [a, c, c + along[:, 0], c + along[:, 1]]
        side = (1.0, -1.0, -1.0, -1.0)
    pts = np.stack(p, 1)
    move = rng.uniform(-1.0, 2.0, n) * dist / 2
    disp = np.stack([s * normal * move[:, None] for s in side], 1) + rng.normal(0, 0.1, (n, 4, 3)) * dist[:, None, None]
    return np.ascontiguousarray(pts.reshape(n, 12)), np.ascontiguousarray(disp.reshape(n, 12)), dist * dist


def prepare(case, seed):
    if case["kind"] == "mlp":
        X, T = _rows(case, seed)
        return {"case": case, "net": WarmStartMLP(params=_weights()), "X": X, "T": T}
    if case["kind"] == "ccd":
        pts, disp, d2 = _pairs(case, seed)
        return {"case": case, "pts": pts, "disp": disp, "d2": d2, "toc": np.zeros(case["pairs"])}
    state = _sim(case, seed) | {"case": case}
    if case.get("warm") or case["kind"] == "predict":
        state["warm"] = LearnedWarmStart(WarmStartMLP(params=_weights()), scale_for(state["scene"]))
    if case["kind"] == "predict":
        state["sim"].find_constraints()
    return state


# ---- one pass ---------------------------------------------------------------
def _step(st):
    sim = st["sim"]
    sim.set_state(st["x"], st["v"])
    sim.frame = st["frame"]
    for _ in range(st["case"]["steps"]):
        sim.step(st.get("warm"))
    return {"x": sim.x, "v": sim.v}


def _direction(st):
    sim = st["sim"]
    sim.apply_sol(0.0)  # x is written between two directions of a step
    counts = sim.find_constraints()
    sim.compute_hessian_and_gradient()
    sim.solve_system(tol=sim.pcg_tol_search)
    if st["case"]["fp32"]:
        sim.refine_solve()
    done = sim.output_residual() < sim.setup.newton_tol  # the Newton test
    return {"counts": np.array(counts), "done": int(done), "rhs": sim.vector(2), "direction": sim.vector(1)}


def _linesearch(st):
    sim = st["sim"]
    sim.apply_sol(0.0)  # back to the start of the search
    before = sim.find_constraints()
    E0, parts0 = sim.compute_energy(parts=True)
    sim.save_xPrev()
    alpha, bounds = sim.compute_intersection_free_step_size(parts=True)
    sim.apply_sol(alpha)
    hits = sim.check_collision()
    after = sim.find_constraints()
    E, parts = sim.compute_energy(parts=True)
    return {"counts": np.array([before, after]), "hits": hits, "inertia0": float(parts0[0]),
            "elastic0": float(parts0[1]), "barrier0": float(parts0[2]), "E0": E0, "alpha": alpha, "bounds": bounds,
            "parts": parts, "E": E, "x": sim.x}


def _predict(st):
    st["warm"](st["sim"])
    return {"increment": st["sim"].vector(1)}


def _mlp(st):
    if st["case"]["backward"]:
        loss, grad = st["net"].grad(st["X"], st["T"])
        return {"loss": np.float32(loss), "grad": grad}
    return {"out": st["net"].forward(st["X"])}


def _ccd(st):
    c = st["case"]
    _lib.call("fipc_batch_ccd", int(c["edges"]), c["pairs"], _lib.dptr(st["pts"]), _lib.dptr(st["disp"]), 0.2,
              _lib.dptr(st["d2"]), _lib.dptr(st["toc"]))
    return {"toc": st["toc"]}


RUN = {"step": _step, "direction": _direction, "linesearch": _linesearch, "predict": _predict, "mlp": _mlp,
       "ccd": _ccd}


def run(state):
    return RUN[state["case"]["kind"]](state)


# ---- compulsory work --------------------------------------------------------
def _sizes(case):
    """vertices, tets, and stored upper blocks (7.3 a vertex on these lattices)"""
    if case["scene"] == "slab":
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        v, t = nx * ny * nz + 16, 5 * ((nx - 1) * (ny - 1) * (nz - 1) + 2)
    else:
        cubes = case["m"] ** 2 * case["layers"]
        v, t = cubes * case["n"] ** 3 + 8, 5 * (cubes * (case["n"] - 1) ** 3 + 1)
    return v, t, v + t * 1.232


def _direction_work(case, iterations):
    """One assembly (tet data and positions read, block values and gradient
    written) and the iterations of conjugate gradients (block values, indices,
    the product's two vectors, and the update's)."""
    v, t, b = _sizes(case)
    s = 4 if case["fp32"] else 8
    nbytes = t * 112 + v * 24 + b * 9 * s + v * 24
    nbytes += iterations * (b * (9 * s + 4) + (b - v) * 8 + v * (8 + 6 * s) + v * (42 * s + 1))
    return nbytes, t * 5000 + iterations * (2 * b - v) * 18


def work(case):
    kind = case["kind"]
    params = NET[0] * NET[1] + (NET[2] - 1) * NET[1] ** 2 + NET[1] * NET[3]
    if kind == "mlp":
        n = case["rows"]
        return {"bytes": n * 4 * (NET[0] + NET[3]) + params * (8 if case["backward"] else 4),
                "flops": n * params * (6 if case["backward"] else 2)}
    if kind == "ccd":
        # about 9,500 operations a pair: two root isolations
        return {"bytes": case["pairs"] * 208, "flops": case["pairs"] * 9500}
    v, t, _ = _sizes(case)
    if kind == "predict":
        return {"bytes": v * (12 * 8 + 1 + 24), "flops": v * params * 2}
    # the line search reads tets and positions for two energies and the
    # inversion bound
    search = {"bytes": 2 * (t * 112 + v * 56) + t * 16 + v * 48, "flops": t * 700}
    if kind == "linesearch":
        return search
    # about 50 iterations to 1e-6
    nbytes, flops = _direction_work(case, 50)
    if kind == "direction":
        return {"bytes": nbytes, "flops": flops}
    # two to three Newton iterations a step; the FP32 form solves most of them loosely
    loose, its = _direction_work(case, 22 if case["fp32"] else 50)
    return {"bytes": case["steps"] * 2.2 * (loose + search["bytes"]) + v * 96,
            "flops": case["steps"] * 2.2 * (its + search["flops"])}


# ---- the same in 64 bits ----------------------------------------------------
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _exact_mlp(case, seed):
    X, T = (torch.from_numpy(a).double() for a in _rows(case, seed))
    w = torch.from_numpy(_weights().copy()).double().requires_grad_(case["backward"])
    dims, o, h = [NET[0]] + [NET[1]] * NET[2] + [NET[3]], 0, X
    for k in range(len(dims) - 1):
        a, b = dims[k], dims[k + 1]
        h = h @ w[o:o + a * b].reshape(a, b) + w[o + a * b:o + a * b + b]
        o += a * b + b
        if k < len(dims) - 2:
            h = torch.nn.functional.silu(h)
    if not case["backward"]:
        return {"out": h}
    loss = ((h - T) ** 2).mean()
    return {"loss": loss.detach(), "grad": torch.autograd.grad(loss, w)[0]}


class _Elastic:
    """Rest shapes, masses and deformation gradients of a state."""

    def __init__(self, case, seed):
        sc = _scene(case)
        x, v, _, frame = _state(case, sc, seed)
        dev = _device()
        self.free, self.dt = torch.from_numpy(~sc.dirichlet_mask).to(dev), sc.dt
        self.x, rest = torch.from_numpy(x).to(dev), torch.from_numpy(sc.x).to(dev)
        t = self.t = torch.from_numpy(sc.tets.astype(np.int64)).to(dev)
        self.rest = rest
        dm = torch.stack([rest[t[:, k]] - rest[t[:, 0]] for k in (1, 2, 3)], 2)
        ds = torch.stack([self.x[t[:, k]] - self.x[t[:, 0]] for k in (1, 2, 3)], 2)
        self.vol = (dm[:, :, 0] * torch.linalg.cross(dm[:, :, 1], dm[:, :, 2])).sum(1) / 6
        # rows of the inverse: cross products of the columns over the determinant
        self.inv = torch.stack([torch.linalg.cross(dm[:, :, (j + 1) % 3], dm[:, :, (j + 2) % 3]) for j in range(3)],
                               1) / (6 * self.vol)[:, None, None]
        self.F = (ds[:, :, :, None] * self.inv[:, None]).sum(2)
        E, nu = torch.from_numpy(sc.youngs).to(dev), torch.from_numpy(sc.poisson).to(dev)
        self.la, self.mu = E * nu / ((1 + nu) * (1 - 2 * nu)), E / (2 * (1 + nu))
        F = self.F
        self.cof = torch.stack([torch.linalg.cross(F[:, (i + 1) % 3], F[:, (i + 2) % 3]) for i in range(3)], 1)
        self.J = (F[:, 0] * self.cof[:, 0]).sum(1)
        self.mass = torch.zeros(len(x), dtype=torch.float64, device=dev)
        for k in range(4):
            self.mass.index_add_(0, t[:, k], self.vol * torch.from_numpy(sc.density).to(dev) / 4)
        # x moved by dt v in the step before, so the next inertial increment
        # is x - (x - dt v) + dt^2 g; the fixed vertices go to new positions
        inc = x - (x - sc.dt * v)
        inc[:, 1] += sc.dt * sc.dt * sc.gravity
        inc[sc.dirichlet_mask] = sc.dirichlet_rows(frame * sc.dt)[1] - x[sc.dirichlet_mask]
        self.inc = torch.from_numpy(inc).to(dev)


def _exact_linesearch(case, seed):
    """The inertia and the elastic energy at the start of the search."""
    e = _Elastic(case, seed)
    logj = torch.log(e.J)
    psi = e.mu / 2 * ((e.F * e.F).sum((1, 2)) - 3) - e.mu * logj + e.la / 2 * logj ** 2
    inertia = 0.5 * (e.mass * (e.inc ** 2).sum(1)).sum()
    none = dict.fromkeys(("counts", "hits", "barrier0", "E0", "alpha", "bounds", "parts", "E", "x"))
    return none | {"inertia0": float(inertia), "elastic0": float((psi * e.vol).sum() * e.dt * e.dt)}


def _dot(a, b):
    return (a * b).sum(-1)


def _cross(a, b):
    return torch.linalg.cross(a, b)


# squared distances, of points p[..., k, 3]
def _point_point(p):
    return _dot(p[..., 0, :] - p[..., 1, :], p[..., 0, :] - p[..., 1, :])


def _point_line(p):
    n, e = _cross(p[..., 1, :] - p[..., 0, :], p[..., 2, :] - p[..., 0, :]), p[..., 2, :] - p[..., 1, :]
    return _dot(n, n) / _dot(e, e)


def _point_plane(p):
    n = _cross(p[..., 2, :] - p[..., 1, :], p[..., 3, :] - p[..., 1, :])
    return _dot(p[..., 0, :] - p[..., 1, :], n) ** 2 / _dot(n, n)


def _line_line(p):
    n = _cross(p[..., 1, :] - p[..., 0, :], p[..., 3, :] - p[..., 2, :])
    return _dot(p[..., 2, :] - p[..., 0, :], n) ** 2 / _dot(n, n)


def _near(lo_a, hi_a, lo_b, hi_b, dh):
    """Index pairs of boxes that overlap within dh."""
    out, step = [], max(1, 200_000_000 // max(1, len(lo_b)))
    for i in range(0, len(lo_a), step):
        ok = torch.ones(len(lo_a[i:i + step]), len(lo_b), dtype=torch.bool, device=lo_a.device)
        for d in range(3):
            ok &= lo_a[i:i + step, None, d] < hi_b[None, :, d] + dh
            ok &= lo_b[None, :, d] - dh < hi_a[i:i + step, None, d]
        a, b = torch.nonzero(ok, as_tuple=True)
        out.append(torch.stack([a + i, b]))
    return torch.cat(out, 1)


def _point_triangle_type(p):
    """0-2 a vertex, 3-5 an edge, 6 the face of the triangle nearest to the point."""
    P, T = p[:, 0], [p[:, 1], p[:, 2], p[:, 3]]
    n = _cross(T[1] - T[0], T[2] - T[0])
    s, side = [], []
    for k in range(3):
        e, d = T[(k + 1) % 3] - T[k], P - T[k]
        s.append(_dot(e, d) / _dot(e, e))
        side.append(_dot(_cross(e, n), d))
    kind = torch.full((len(p),), 6, device=p.device)
    for k in (2, 1, 0):  # vertex k: before edge k's start, past the previous edge's end
        kind = torch.where((s[k] <= 0) & (s[(k + 2) % 3] >= 1), k, kind)
    for k in (2, 1, 0):
        beyond = side[k] > 0 if k == 2 else side[k] >= 0
        kind = torch.where((s[k] > 0) & (s[k] < 1) & beyond, 3 + k, kind)
    return kind


def _edge_edge_type(p):
    """3 i + j: the nearest features of two edges, i (j) = 0, 1 the ends, 2 the inside of the first (second)."""
    u, v, w = p[:, 1] - p[:, 0], p[:, 3] - p[:, 2], p[:, 0] - p[:, 2]
    a, b, c, d, e = _dot(u, u), _dot(u, v), _dot(v, v), _dot(u, w), _dot(v, w)
    D = a * c - b * b
    sN, n = b * e - c * d, _cross(u, v)
    parallel = (sN > 0) & (sN < D) & (a * e - b * d > 0) & (a * e - b * d < D) & \
        ((_dot(n, w) == 0) | (_dot(n, n) < 1e-20 * a * c))
    start, end = (sN <= 0) | (parallel & (sN < D / 2)), (sN >= D) | (parallel & (sN >= D / 2))
    end &= ~start
    tN = torch.where(start, e, torch.where(end, e + b, a * e - b * d))
    tD = torch.where(start | end, c, D)
    i = torch.where(start, 0, torch.where(end, 1, 2))
    low, high = tN <= 0, tN >= tD
    q = torch.where(low, -d, -d + b)
    i = torch.where(low | high, torch.where(q <= 0, 0, torch.where(q >= a, 1, 2)), i)
    return 3 * i + torch.where(low, 0, torch.where(high, 1, 2))


def _contacts(e, sc):
    """(distance, vertices of the row, places of the distance's points in it,
    mollified) for every kind of contact within the barrier distance, rows unique."""
    x, dh, dev = e.x, sc.dhat, e.x.device
    points, edges, tris = (torch.from_numpy(a.astype(np.int64)).to(dev) for a in sc.boundary)
    rows = {}

    def add(name, ids):
        rows.setdefault(name, []).append(ids)

    lo, hi = x[tris].amin(1), x[tris].amax(1)
    a, b = _near(x[points], x[points], lo, hi, dh)
    q = torch.cat([points[a][:, None], tris[b]], 1)
    q = q[(q[:, 1:] != q[:, :1]).all(1)]
    kind = _point_triangle_type(x[q])
    for k in range(7):
        c = q[kind == k]
        if k < 3:
            c, f, name = c[:, [0, 1 + k]], _point_point, "pp"
        elif k < 6:
            c, f, name = c[:, [0, 1 + k - 3, 1 + (k - 2) % 3]], _point_line, "pe"
        else:
            f, name = _point_plane, "pt"
        add(name, c[f(x[c]) < dh * dh])
    lo, hi = x[edges].amin(1), x[edges].amax(1)
    a, b = _near(lo, hi, lo, hi, dh)
    q = torch.cat([edges[a], edges[b]], 1)[a < b]
    q = q[(q[:, :2, None] != q[:, None, 2:]).all(2).all(1)]
    kind = _edge_edge_type(x[q])
    n, r = _cross(x[q[:, 1]] - x[q[:, 0]], x[q[:, 3]] - x[q[:, 2]]), e.rest
    moll = _dot(n, n) < 1e-3 * _point_point(r[q[:, :2]]) * _point_point(r[q[:, 2:]])
    for k in range(9):
        i, j = divmod(k, 3)
        c, m = q[kind == k], moll[kind == k]
        if i < 2 and j < 2:
            c, at, f, name = c[:, [i, 1 - i, 2 + j, 3 - j]], [0, 2], _point_point, "pp"
        elif i < 2:
            c, at, f, name = c[:, [i, 1 - i, 2, 3]], [0, 2, 3], _point_line, "pe"
        elif j < 2:
            c, at, f, name = c[:, [2 + j, 3 - j, 0, 1]], [0, 2, 3], _point_line, "pe"
        else:
            at, f, name = [0, 1, 2, 3], _line_line, "ee"
        near = f(x[c[:, at]]) < dh * dh
        add(name, c[near & ~m][:, at])
        add(name + "m", c[near & m])
    form = {"pp": (_point_point, [0, 1], False), "pe": (_point_line, [0, 1, 2], False),
            "pt": (_point_plane, [0, 1, 2, 3], False), "ee": (_line_line, [0, 1, 2, 3], False),
            "ppm": (_point_point, [0, 2], True), "pem": (_point_line, [0, 2, 3], True),
            "eem": (_line_line, [0, 1, 2, 3], True)}
    for name, parts in rows.items():
        ids = torch.cat(parts)
        if len(ids):
            f, at, m = form[name]
            yield f, torch.unique(ids, dim=0), at, m


def _kappa(sc, mass):
    """The barrier's stiffness of a scene, from its mean mass."""
    h, d = sc.dhat ** 2, 1e-16
    second = (-2 * math.log(d / h) - 4 * (d - h) / d) + ((d - h) / d) ** 2
    return 10 * 1e13 * float(mass.mean()) / (4e-16 * second)


def _contact_terms(e, sc):
    """(vertices, gradient, projected Hessian) of every contact row."""
    h, kappa = sc.dhat ** 2, _kappa(sc, e.mass)
    for f, ids, at, moll in _contacts(e, sc):
        k = ids.shape[1]

        def energy(p, eps):
            p = p.reshape(k, 3)
            d = f(p[at])
            b = -kappa * (d - h) ** 2 * torch.log(d / h)
            if moll:
                n = _cross(p[1] - p[0], p[3] - p[2])
                r = _dot(n, n) / eps
                b = b * (2 - r) * r
            return b

        p, rest = e.x[ids].reshape(-1, 3 * k), e.rest[ids]
        eps = 1e-3 * _point_point(rest[:, :2]) * _point_point(rest[:, 2:]) if moll else torch.ones_like(p[:, 0])
        g = torch.func.vmap(torch.func.grad(energy))(p, eps)
        H = torch.func.vmap(torch.func.hessian(energy))(p, eps)
        lam, V = np.linalg.eigh(((H + H.transpose(1, 2)) / 2).cpu().numpy())
        H = (V * np.maximum(lam, 0)[:, None, :]) @ V.transpose(0, 2, 1)
        yield ids, g, torch.from_numpy(H).to(p.device)


def _elastic_hessians(e):
    """The projected 12 x 12 Hessians of the tets: the Hessian over the
    singular values is projected, and each 2 x 2 twist block by its closed
    form, which for a negative smaller eigenvalue keeps b^2 / (a + |b|)."""
    lam, V = np.linalg.eigh((e.F.transpose(1, 2)[..., None] * e.F[:, None]).sum(2).cpu().numpy())
    V = torch.from_numpy(V).to(e.F.device)
    U = (e.F[:, :, :, None] * V[:, None]).sum(2)
    s = torch.sqrt((U * U).sum(1))
    U = U / s[:, None]
    lp, la, mu = torch.log(e.J), e.la, e.mu
    M = torch.zeros(len(s), 9, 9, dtype=torch.float64, device=s.device)
    S = la[:, None, None] / (s[:, :, None] * s[:, None, :])
    S[:, range(3), range(3)] = mu[:, None] * (1 + s ** -2) - la[:, None] * s ** -2 * (lp[:, None] - 1)
    minor = S[:, 0, 0] * S[:, 1, 1] - S[:, 0, 1] ** 2
    det = (S[:, 0] * _cross(S[:, 1], S[:, 2])).sum(1)
    bad = torch.nonzero((S[:, 0, 0] <= 0) | (minor <= 0) | (det <= 0))[:, 0]
    if len(bad):
        w, Q = np.linalg.eigh(S[bad].cpu().numpy())
        S[bad] = torch.from_numpy((Q * np.maximum(w, 0)[:, None]) @ Q.transpose(0, 2, 1)).to(s.device)
    for i in range(3):
        for j in range(3):
            M[:, 4 * i, 4 * j] = S[:, i, j]
    g = mu[:, None] * (s - 1 / s) + la[:, None] / s * lp[:, None]
    for i, j in ((0, 1), (1, 2), (2, 0)):
        left = (mu + (mu - la * lp) / (s[:, i] * s[:, j])) / 2
        right = (g[:, i] + g[:, j]) / (2 * (s[:, i] + s[:, j]))
        a, b = left + right, left - right
        cut = a - b.abs() < 0
        c = torch.where(cut, b * b / (a + b.abs()), a)
        d = torch.where(cut, c * torch.sign(b), b)
        p, q = 3 * i + j, 3 * j + i
        M[:, p, p], M[:, q, q], M[:, p, q], M[:, q, p] = c, c, d, d
    # vertex a's share of w_(k,l) = u_k v_l^T: sum_j B[a][j] V[j][l] times U[:, k]
    B = torch.cat([-e.inv.sum(1, keepdim=True), e.inv], 1)
    BV = (B[:, :, :, None] * V[:, None]).sum(2)
    Z = (U[:, None, :, :, None] * BV[:, :, None, None, :]).reshape(len(s), 12, 9)
    return (Z @ M) @ Z.transpose(1, 2).contiguous() * (e.dt ** 2 * e.vol)[:, None, None]


def _exact_direction(case, seed):
    """The right-hand side and the solution of the projected Newton system,
    by conjugate gradients in 64 bits to the end of their accuracy."""
    e, sc = _Elastic(case, seed), _scene(case)
    nv, dev = len(e.x), e.x.device
    P = e.mu[:, None, None] * e.F + ((e.la * torch.log(e.J) - e.mu) / e.J)[:, None, None] * e.cof
    B = torch.cat([-e.inv.sum(1, keepdim=True), e.inv], 1)
    g = (P[:, None] * B[:, :, None, :]).sum(3) * (e.dt ** 2 * e.vol)[:, None, None]
    terms = [(e.t, g.reshape(-1, 12), _elastic_hessians(e))] + list(_contact_terms(e, sc))
    b = e.mass[:, None] * e.inc
    D = torch.zeros(nv, 3, 3, dtype=torch.float64, device=dev)
    D[:, range(3), range(3)] = e.mass[:, None]
    for ids, gr, H in terms:
        k = ids.shape[1]
        b = b.index_add(0, ids.reshape(-1), -gr.reshape(-1, 3))
        H4 = H.reshape(-1, k, 3, k, 3)
        for a in range(k):
            D.index_add_(0, ids[:, a], H4[:, a, :, a])
    free = e.free[:, None].double()
    rhs = b * free

    def product(p):
        q = e.mass[:, None] * p
        for ids, _, H in terms:
            q = q.index_add(0, ids.reshape(-1), (H * p[ids].reshape(len(ids), 1, -1)).sum(2).reshape(-1, 3))
        return q * free

    inv = torch.linalg.inv(D.cpu()).to(dev)
    fixed = e.inc * (1 - free)
    r = rhs - product(fixed)
    x, goal = torch.zeros_like(r), float((r * r).sum()) * 1e-26
    for _ in range(3):  # restarts with the true residual
        z = (inv * r[:, None]).sum(2) * free
        p, rz = z, (r * z).sum()
        for it in range(4000):
            q = product(p)
            alpha = rz / (p * q).sum()
            x, r = x + alpha * p, r - alpha * q
            if it % 16 == 15 and float((r * r).sum()) < goal:
                break
            z = (inv * r[:, None]).sum(2) * free
            new = (r * z).sum()
            p, rz = z + (new / rz) * p, new
        r = rhs - product(fixed + x)
    x = x + fixed
    return {"counts": None, "done": None, "rhs": rhs.cpu(), "direction": x.cpu()}


def exact(case, seed):
    """The network, the directions, and the parts of the energy that need no
    contact search.  A step ends wherever its Newton tolerance lets it, a time
    of impact is a conservative bound, and the warm start's features are not
    restated here."""
    kind = case["kind"]
    if kind == "mlp":
        return _exact_mlp(case, seed)
    if kind == "linesearch":
        return _exact_linesearch(case, seed)
    if kind == "direction":
        return _exact_direction(case, seed)
    return None
