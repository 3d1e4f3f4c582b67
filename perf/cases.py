"""The measured work of the framework: what a DEM user runs, through the public entry points.

Sphere and polyhedra simulations through the fused engine (xdem_run_steps) and operator by operator, each pass
a block of time steps followed by the frame a program keeps (state per particle id, in host memory), and the
learned surrogate: inference, one training window, and a drift-checked run. Sizes and parameters are those of
the configurations, the tests and the benchmark: the walled deposition, the periodic polydisperse packing at
solid fraction 0.55, the polyhedra bed, the triangle mesh, the shipped surrogate networks.

`exact` restates each path in plain torch at 64 bits, with its own neighbour search and summation order.
"""
import math

import numpy as np
import torch

from exadem_amd import inputs, native, stl, surrogate
from exadem_amd.sim import PolySim, SphereSim, scheme

DEV = "cuda" if torch.cuda.is_available() else "cpu"

FRAME = {"position": ("rx", "ry", "rz"), "velocity": ("vx", "vy", "vz"), "spin": ("vrotx", "vroty", "vrotz"),
         "orientation": ("qw", "qx", "qy", "qz"), "acceleration": ("fx", "fy", "fz")}
ROWS = [k for names in FRAME.values() for k in names]
WEIGHTS = {10: surrogate.WEIGHTS, 100: surrogate.WEIGHTS_K100, 200: surrogate.WEIGHTS_K200}


# ------------------------------------------------------------------------------------------------ cases
def listed():
    return [
        # a small walled sample, as in parameter sweeps and calibration runs: latency and launches decide
        {"name": "deposition_1k", "kind": "deposition", "n": 997, "steps": 200, "form": "fp64", "path": "engine"},
        # the plain deposition configuration at its own size
        {"name": "deposition_10k", "kind": "deposition", "n": 10000, "steps": 200, "form": "fp64", "path": "engine"},
        # the same path operator by operator, as decks and coupled programs drive it
        {"name": "operators_30k", "kind": "deposition", "n": 30011, "steps": 25, "form": "fp64", "path": "operators"},
        # a periodic flow with a large time step: the neighbour lists are rebuilt every few dozen steps
        {"name": "flow_120k", "kind": "flow", "n": 120001, "steps": 200, "form": "fp64", "path": "engine"},
        # the benchmark packing, plain form
        {"name": "periodic_1m", "kind": "periodic", "n": 1000000, "steps": 100, "form": "fp64", "path": "engine"},
        # the benchmark packing, FP32-force form
        {"name": "periodic_fp32_700k", "kind": "periodic", "n": 700001, "steps": 100, "form": "fp32", "path": "engine"},
        # a bed on a triangulated floor
        {"name": "mesh_150k", "kind": "mesh", "n": 150003, "steps": 100, "form": "fp64", "path": "engine"},
        # the relaxed polyhedra bed of the benchmark
        {"name": "poly_bed_200k", "kind": "poly_bed", "n": 200000, "steps": 100},
        # a moving polyhedra bed: contacts of every type and list rebuilds
        {"name": "poly_flow_20k", "kind": "poly_flow", "n": 20011, "steps": 100},
        # one inference of the shipped network on a packing
        {"name": "gnn_forward_500k", "kind": "forward", "n": 500009, "substeps": 100},
        # one training window at the size of the training runs
        {"name": "gnn_train_50k", "kind": "train", "n": 50000, "substeps": 10},
        # a drift-checked surrogate run: 19 network steps and one checked window of DEM steps
        {"name": "surrogate_200k", "kind": "surrogate", "n": 200000, "substeps": 10, "steps": 20},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["deposition", "deposition", "operators", "flow", "periodic", "periodic", "mesh", "poly_bed",
                       "poly_flow", "forward", "train", "surrogate"])
    form = rng.choice(["fp64", "fp64", "fp32"])
    if kind == "deposition":
        return {"kind": kind, "n": _log(rng, 500, 100000), "steps": rng.randint(50, 200), "form": form, "path": "engine"}
    if kind == "operators":
        return {"kind": "deposition", "n": _log(rng, 1000, 100000), "steps": rng.randint(10, 25), "form": form,
                "path": "operators"}
    if kind == "flow":
        return {"kind": kind, "n": _log(rng, 5000, 120000), "steps": rng.randint(100, 200), "form": form,
                "path": "engine"}
    if kind == "periodic":
        return {"kind": kind, "n": _log(rng, 5000, 1000000), "steps": rng.randint(50, 100), "form": form,
                "path": "engine"}
    if kind == "mesh":
        return {"kind": kind, "n": _log(rng, 10000, 150000), "steps": rng.randint(50, 100), "form": form,
                "path": "engine"}
    if kind in ("poly_bed", "poly_flow"):
        return {"kind": kind, "n": _log(rng, 1000, 200000 if kind == "poly_bed" else 40000), "steps": rng.randint(40, 100)}
    if kind == "forward":
        return {"kind": kind, "n": _log(rng, 5000, 500000), "substeps": rng.choice([10, 100, 200])}
    if kind == "train":
        return {"kind": kind, "n": _log(rng, 4000, 60000), "substeps": rng.choice([10, 10, 20])}
    return {"kind": kind, "n": _log(rng, 20000, 200000), "substeps": 10, "steps": 20}


# ------------------------------------------------------------------------------------------------ inputs
def _split(tiles):
    """tiles = a * b * c with near-equal factors."""
    a = max(1, int(round(tiles ** (1.0 / 3.0))))
    b = max(1, int(round(math.sqrt(tiles / a))))
    return a, b, max(1, int(math.ceil(tiles / (a * b))))


def _packing(n, seed, v_mean=(0.0, 0.0, 0.0), sigma=0.1, spin=0.0, dt=5e-6, gravity=(0.0, 0.0, -9.81)):
    """n polydisperse spheres (radius U[0.5, 1], solid fraction 0.55, periodic): a relaxed periodic tile of a few
    thousand spheres repeated, each sphere displaced a little, with velocities (and spins) of its own. The few spheres above n are
    left out at random."""
    a, b, c = _split(max(1, n // 5000))
    m = -(-n // (a * b * c))
    t = inputs.polydisperse(n=m, seed_radius=seed + 1, seed_vel=seed + 2, seed_pos=seed + 3, relax_sweeps=150)
    rng = np.random.default_rng(seed)
    box = np.array(t.domain.hi[:])
    g = np.stack(np.meshgrid(np.arange(a), np.arange(b), np.arange(c), indexing="ij"), -1).reshape(-1, 3)
    off = (g * box)[:, None, :]
    x = (np.stack([t.particles[k] for k in ("rx", "ry", "rz")], 1)[None] + off).reshape(-1, 3)
    r = np.tile(t.particles["radius"], len(g))
    keep = np.ones(len(r), bool)
    keep[rng.choice(len(r), len(r) - n, replace=False)] = False
    # the relaxation leaves pairs that touch to the last bit, and a contact's damping sets in at once
    x, r = x[keep] + rng.normal(0.0, 1e-4, (n, 3)), r[keep]
    v = rng.normal(0.0, sigma, (3, n)) + np.array(v_mean)[:, None]
    p = inputs.sphere_set(x[:, 0], x[:, 1], x[:, 2], r, 2500.0, v[0], v[1], v[2])
    if spin > 0:
        w = rng.normal(0.0, spin, (3, n))
        p["vrotx"], p["vroty"], p["vrotz"] = (np.ascontiguousarray(w[i]) for i in range(3))
    dom = native.domain((0.0, 0.0, 0.0), tuple(box * np.array([a, b, c])), (True, True, True), 2.1)
    cp = native.contact_params(kn=1e5, mu=0.3, damp_rate=0.9)
    return inputs.Workload("packing", p, dom, [], cp, cp, dt, 0, 0.1, gravity)


def _deposition(n, seed):
    """A contact-rich deposition in a walled box of the configuration's proportions (1 : 1 : 2), the bed on the
    floor and against the side walls."""
    side = max(4, int(math.ceil((n / 1.5) ** (1.0 / 3.0))))
    edge = 0.98 * (side - 1) + 0.96
    return inputs.deposition(n=n, spacing=0.98, jitter=0.05, seed=seed + 1, start=0.48, box=(edge, edge, 2.0 * edge + 2.0))


def _floor(w):
    """A triangulated floor of the box: spacing about 2, two triangles per square."""
    hi = np.array(w.domain.hi[:])
    gx = np.linspace(0.0, hi[0], max(2, int(hi[0] // 2) + 1))
    X, Y = np.meshgrid(gx, gx, indexing="ij")
    P = np.stack([X, Y, np.zeros_like(X)], -1)
    A, B, C, D = P[:-1, :-1], P[1:, :-1], P[1:, 1:], P[:-1, 1:]
    tri = np.stack([np.stack([A, B, C], -2), np.stack([A, C, D], -2)], -3).reshape(-1, 3, 3)
    v, e, f = stl.build_shape(tri)
    return {"mesh_id": 0, "vertices": v, "edges": e, "faces": f, "minkowski": 0.01}


def _poly(n, seed, moving):
    """Cubes and octahedra at solid fraction 0.45 (the benchmark's growth on a tile, repeated along the periodic
    axes); moving: a mean velocity along x with fluctuations, at a time step that brings contacts and rebuilds."""
    a = max(1, int(round(math.sqrt(n / 1000.0))))
    b = max(1, n // (1000 * a))
    m = -(-n // (a * b))
    t = inputs.polyhedra_dense(n=m, phi=0.45, seed=seed + 1, dt=2e-4 if moving else 2e-6)
    rng = np.random.default_rng(seed)
    hi = np.array(t.domain.hi[:])
    g = np.stack(np.meshgrid(np.arange(a), np.arange(b), indexing="ij"), -1).reshape(-1, 2)
    p = {k: np.tile(v, len(g)) for k, v in t.particles.items()}
    p["rx"] = p["rx"] + np.repeat(g[:, 0] * hi[0], m)
    p["ry"] = p["ry"] + np.repeat(g[:, 1] * hi[1], m)
    keep = np.ones(len(p["rx"]), bool)
    keep[rng.choice(len(keep), len(keep) - n, replace=False)] = False
    p = {k: np.ascontiguousarray(v[keep]) for k, v in p.items()}
    p["id"] = np.arange(n, dtype=np.uint64)
    if moving:
        v = rng.normal(0.0, 0.3, (3, n))
        v[0] += 4.0
        p["vx"], p["vy"], p["vz"] = (np.ascontiguousarray(v[i]) for i in range(3))
    dom = native.domain((0.0, 0.0, 0.0), (hi[0] * a, hi[1] * b, hi[2]), (True, True, False), t.domain.cell_size)
    w = inputs.Workload("polyhedra", p, dom, t.walls, t.cp, t.cpd, t.dt, 0, t.rcut_inc, t.gravity)
    w.shapes = t.shapes
    return w


def _workload(case, seed):
    kind, n = case["kind"], case["n"]
    if kind == "deposition":
        return _deposition(n, seed)
    if kind == "mesh":  # the same bed on a triangulated floor in place of the plane
        w = _deposition(n, seed)
        w.walls = [wl for wl in w.walls if wl["offset"] != 0.0 or wl["normal"][2] == 0.0]
        return w
    if kind == "flow":  # plug flow without gravity: the mean velocity, and with it the rebuild rate, stays
        return _packing(n, seed, v_mean=(8.0, 2.0, 0.0), sigma=0.3, dt=1e-4, gravity=(0.0, 0.0, 0.0))
    if kind in ("poly_bed", "poly_flow"):
        return _poly(n, seed, kind == "poly_flow")
    if kind in ("forward", "train"):
        return _packing(n, seed, spin=0.1)
    if kind == "surrogate":  # no mean acceleration: the run stays near the packings that the network knows
        return _packing(n, seed, spin=0.1, gravity=(0.0, 0.0, 0.0))
    return _packing(n, seed)


def _pinned(shape, dtype):
    return torch.zeros(shape, dtype=dtype, pin_memory=DEV == "cuda")


def prepare(case, seed):
    kind, n = case["kind"], case["n"]
    w = _workload(case, seed)
    st = {"case": case, "ids": _pinned(n, torch.int64), "n": n}
    if kind.startswith("poly"):
        st["sim"] = PolySim(w)
    else:
        form = native.XDEM_FORM_FP32 if case.get("form") == "fp32" else native.XDEM_FORM_FP64
        st["sim"] = SphereSim(w, form=form, mesh=_floor(w) if kind == "mesh" else None)
    sim = st["sim"]
    sim.first_iteration()
    arrays = {"id": st["ids"].numpy().view(np.uint64)}
    if kind in ("forward", "train", "surrogate"):
        params, scales = surrogate.load(WEIGHTS.get(case["substeps"], surrogate.WEIGHTS))
        scales = dict(scales, substeps=case["substeps"])
        if kind == "train":
            params = surrogate.init_params(seed)
        if kind != "forward":
            surrogate.settle(sim, case["substeps"])
        st["gnn"] = surrogate.attach(sim.ctx, params, scales, train=kind == "train")
        st["scheme"] = scheme(w)
    if kind == "forward":
        st["raw"] = _pinned((n, 6), torch.float32)
    elif kind == "train":
        st["grads"] = _pinned(native.GNN_NPARAMS, torch.float32)
        st["params"] = _pinned(native.GNN_NPARAMS, torch.float32)
    else:
        st["raw"] = _pinned((len(ROWS), n), torch.float64)
        arrays.update({k: st["raw"][i].numpy() for i, k in enumerate(ROWS)})
    st["fields"] = native.particles_struct(arrays, n)
    if "raw" in st:
        st["dev"] = torch.empty_like(st["raw"], device=DEV, pin_memory=False)
        st["out"] = torch.empty_like(st["dev"])
    sim.ctx.synchronize()
    return st


# ------------------------------------------------------------------------------------------------ one pass
def _frame(st):
    """The state by particle id, as a torch program holds it for analysis (the device keeps particles in cell
    order, and the library hands them over in host arrays: the program's own, pinned)."""
    st["sim"].ctx.call("xdem_particles_download", native.C.byref(st["fields"][0]))
    order = torch.empty(st["n"], dtype=torch.int64, device=DEV)
    order[st["ids"].to(DEV, non_blocking=True)] = torch.arange(st["n"], device=DEV)
    st["dev"].copy_(st["raw"], non_blocking=True)
    if st["case"]["kind"] == "forward":
        return torch.index_select(st["dev"], 0, order, out=st["out"])
    out, at = {}, 0
    torch.index_select(st["dev"], 1, order, out=st["out"])
    for name, rows in FRAME.items():
        out[name] = st["out"][at:at + len(rows)]
        at += len(rows)
    return out


def run(st):
    case, sim = st["case"], st["sim"]
    kind = case["kind"]
    if kind == "forward":
        st["gnn"].call("xdem_gnn_forward", native._ptr(st["raw"].numpy(), native.C.c_float))
        return _frame(st)
    if kind == "train":
        loss, used = st["gnn"].train_window(st["scheme"], 1e-3)
        for name in ("grads", "params"):
            st["gnn"].call("xdem_gnn_get_" + name, native._ptr(st[name].numpy(), native.C.c_float), native.GNN_NPARAMS)
        return {"loss": loss, "used": used, "grads": st["grads"], "params": st["params"]}
    if kind == "surrogate":
        st["gnn"].surrogate_run(st["scheme"], case["steps"], check_every=20, tol=0.01)
    elif case.get("path") == "operators":
        for _ in range(case["steps"]):
            sim.step()
    else:
        sim.run(case["steps"], poll=64)
    return _frame(st)


# ------------------------------------------------------------------------------------------------ cost
def work(case):
    """Bytes: per DEM step each particle's state read and written once and each pair's list word and history (read
    and written) once; per pass the frame. Flops: about 220 per contact and 150 per particle for the DEM, the
    dense and per-edge products of the network (6 list entries per particle)."""
    n, kind = case["n"], case["kind"]
    pairs = 3.0 * n
    row, hist = (256.0, 28.0) if case.get("form") == "fp32" else (300.0, 52.0)
    step_b, step_f = row * n + hist * pairs, 220.0 * pairs + 150.0 * n
    net_f = n * (2.0 * 8 * 128 + 3 * (2.0 * 128 * 256 + 2.0 * 256 * 128 + 6 * 2.0 * 16 * 128) + 2.0 * 128 * 6)
    net_b = n * (128.0 + 24.0 + 6 * 4.0) + 4.0 * native.GNN_NPARAMS
    frame = 8.0 * n * (len(ROWS) + 1)
    if kind.startswith("poly"):  # record read and written, inertia, rebuild reference, about 5 features and 8 entries
        return {"bytes": case["steps"] * n * (256.0 + 24 + 60 + 5 * 12 + 8 * 4) + frame,
                "flops": case["steps"] * n * (5 * 120.0 + 8 * 60 + 150)}
    if kind == "forward":
        return {"bytes": net_b + 32.0 * n, "flops": net_f}
    if kind == "train":
        return {"bytes": net_b + case["substeps"] * step_b + 28.0 * native.GNN_NPARAMS,
                "flops": 3 * net_f + case["substeps"] * step_f}
    if kind == "surrogate":
        return {"bytes": case["steps"] * net_b + case["substeps"] * step_b + frame,
                "flops": case["steps"] * net_f + case["substeps"] * step_f}
    return {"bytes": case["steps"] * step_b + frame, "flops": case["steps"] * step_f}


def tolerance(case):
    kind = case["kind"]
    if kind in ("forward", "train"):  # bfloat16 weights and activations
        return {"rel": 2e-2, "max": 0.5}
    if kind == "surrogate":  # the bfloat16 network's forces act on the state through 19 steps
        return {"rel": 4e-4, "max": 0.1}
    if case.get("form") == "fp32":
        return {"rel": 2e-6, "max": 1e-4}
    return {"rel": 2e-9, "max": 8e-8}


# ------------------------------------------------------------------------------------------------ 64-bit restatement
def _t(a):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device=DEV)


def _dot(a, b):
    return (a * b).sum(-1, keepdim=True)


def _cross(a, b):
    return torch.linalg.cross(a, b)


def _norm(a):
    return torch.sqrt(_dot(a, a))


def _rot(q, v):
    """Rotation of v by the quaternion q (w, x, y, z)."""
    qv = q[..., 1:].expand(v.shape)
    uv = _cross(qv, v)
    return v + 2.0 * (q[..., :1] * uv + _cross(qv, uv))


def _close_pairs(x, cut, lo, hi, per):
    """All i < j closer than cut (minimum image on periodic axes), by cell binning: (i, j)."""
    n = len(x)
    L = hi - lo
    dims = [max(1, int(float(L[a]) // cut)) for a in range(3)]
    xw = x - lo
    for a in range(3):
        if per[a]:
            xw[:, a] = torch.remainder(xw[:, a], L[a])
    cell = torch.stack([(xw[:, a] / L[a] * dims[a]).long().clamp_(0, dims[a] - 1) for a in range(3)], 1)
    cid = (cell[:, 2] * dims[1] + cell[:, 1]) * dims[0] + cell[:, 0]
    order = torch.argsort(cid)
    count = torch.bincount(cid, minlength=dims[0] * dims[1] * dims[2])
    start = torch.cumsum(count, 0) - count
    got = set()
    out_i, out_j = [], []
    me = torch.arange(n, device=x.device)
    for dz in (-1, 0, 1):
        for dy in (-1, 0, 1):
            for dx in (-1, 0, 1):
                key = tuple((d % dims[a]) if per[a] else d for a, d in enumerate((dx, dy, dz)))
                if key in got:  # the same neighbour cell again on a short axis
                    continue
                got.add(key)
                c = cell + torch.tensor([dx, dy, dz], device=x.device)
                ok = torch.ones(n, dtype=torch.bool, device=x.device)
                for a in range(3):
                    if per[a]:
                        c[:, a] = torch.remainder(c[:, a], dims[a])
                    else:
                        ok &= (c[:, a] >= 0) & (c[:, a] < dims[a])
                nid = ((c[:, 2] * dims[1] + c[:, 1]) * dims[0] + c[:, 0]).clamp_(0, len(count) - 1)
                k = torch.where(ok, count[nid], 0)
                i = torch.repeat_interleave(me, k)
                first = torch.repeat_interleave(start[nid] - (torch.cumsum(k, 0) - k), k)
                j = order[first + torch.arange(len(i), device=x.device)]
                d = x[i] - x[j]
                for a in range(3):
                    if per[a]:
                        d[:, a] -= L[a] * torch.round(d[:, a] / L[a])
                sel = (i < j) & ((d * d).sum(1) < cut * cut)
                out_i.append(i[sel])
                out_j.append(j[sel])
    return torch.cat(out_i), torch.cat(out_j)


class _Exact:
    """The time loop at 64 bits. Contacts are lists of (body i, body j or -1, history); subclasses name them."""

    def __init__(self, w):
        p = w.particles
        self.w = w
        self.x, self.v, self.s = (_t(np.stack([p[k] for k in FRAME[f]], 1)) for f in ("position", "velocity", "spin"))
        self.q = _t(np.stack([p[k] for k in FRAME["orientation"]], 1))
        self.m, self.r, self.h = (_t(p[k])[:, None] for k in ("mass", "radius", "homothety"))
        self.I = _t(np.stack([p["inx"], p["iny"], p["inz"]], 1))
        self.lo, self.hi = _t(w.domain.lo[:]), _t(w.domain.hi[:])
        self.per = [bool(v) for v in w.domain.periodic[:]]
        self.L = self.hi - self.lo
        self.g = _t(w.gravity)[None]
        self.wrapped = torch.zeros_like(self.x)  # image shifts applied at rebuilds
        self.hist, self.hold, self.far, self.image = {}, {}, {}, {}
        self.i = self.mesh = self.feat = None
        self.a, self.al = torch.zeros_like(self.x), torch.zeros_like(self.x)
        self.rebuild()

    def shifts(self, i, j):
        """Image shift of j as seen from i."""
        d = self.x[i] - self.x[j]
        s = torch.zeros_like(d)
        for a in range(3):
            if self.per[a]:
                s[:, a] = self.L[a] * torch.round(d[:, a] / self.L[a])
        return s

    def rebuild(self):
        """What a list rebuild does to the state: particles beyond a periodic face are shifted back."""
        y = self.x + self.wrapped
        for a in range(3):
            if self.per[a]:
                self.wrapped[:, a] += torch.where(y[:, a] < self.lo[a], self.L[a], 0.0)
                self.wrapped[:, a] -= torch.where(y[:, a] >= self.hi[a], self.L[a], 0.0)
        self.ref = self.marks()
        self.relist()

    def relist(self):
        """Which contact candidates the lists of a build at the current positions hold (hold[key])."""

    def marks(self):
        return self.x.clone()

    def moved(self):
        return bool(((self.marks() - self.ref).square().sum(-1) >= (0.5 * self.w.rcut_inc) ** 2).any())

    def law(self, cp, meff, dn, n, ci, cj, i, j, ft):
        """Hooke with viscous damping and Coulomb-capped friction: force on i, new history. ci, cj: contact point
        relative to the bodies' centres; j None: a body at rest."""
        vi = self.v[i] - _cross(ci, self.s[i])
        vj = 0.0 if j is None else self.v[j] - _cross(cj, self.s[j])
        vel = vj - vi
        vn = _dot(vel, n)
        fn = torch.clamp(2.0 * cp.damp_rate * torch.sqrt(cp.kn * meff) * vn - cp.kn * dn, min=0.0) * n
        ft = ft + cp.kt * self.w.dt * (vel - vn * n)
        thr = (cp.mu * cp.kn * dn).abs()
        big = _norm(ft)
        ft = torch.where(big > thr, ft * (thr / big.clamp(min=1e-300)), ft)
        return fn + ft, ft

    def add(self, F, M, i, c, f):
        F.index_add_(0, i, f)
        M.index_add_(0, i, _cross(c, f))

    def images(self, key, i, j):
        """At a list rebuild: the candidates whose partner is now a periodic image. Each side of such a pair keeps a
        history of its own (the reference's ghost interactions, keyed by owner and partner): the side of the larger
        id has none when the pair first meets a boundary, and both share one again inside the box."""
        d = self.x[i] + self.wrapped[i] - (self.x[j] + self.wrapped[j])
        now = ((d.abs() > 0.5 * self.L) & torch.tensor(self.per, device=DEV)).any(1)
        if key not in self.image:
            self.far[key] = torch.zeros_like(self.hist[key])
        else:
            fresh = (now & ~self.image[key])[:, None]
            self.far[key] = torch.where(now[:, None], torch.where(fresh, 0.0, self.far[key]), self.hist[key])
        self.image[key] = now

    def pair_contact(self, F, M, key, on, dn, n, ci, cj, i, j, swap=False):
        """Contacts `on` (indices into the candidate list `key`) between bodies i and j (j None: a driver); the
        smaller id is i, or j if swap."""
        hist = self.hist[key]
        cp = self.w.cp if j is not None else self.w.cpd
        meff = self.m[i] if j is None else self.m[i] * self.m[j] / (self.m[i] + self.m[j])
        f, ft = self.law(cp, meff, dn, n, ci, cj, i, j, hist[on])
        hist.zero_()
        hist[on] = ft
        fi = fj = f
        if j is not None:
            far, image = self.far[key], self.image[key][on][:, None]
            f2, ft2 = self.law(cp, meff, dn, n, ci, cj, i, j, far[on])
            f2 = torch.where(image, f2, f)
            far.zero_()
            far[on] = torch.where(image, ft2, ft)
            fi, fj = (f2, f) if swap else (f, f2)
        self.add(F, M, i, ci, fi)
        if j is not None:
            self.add(F, M, j, cj, -fj)

    def walls(self, F, M, pts, rad, body):
        """Planar walls against points of radius rad that belong to bodies `body`."""
        for k, wl in enumerate(self.w.walls):
            nrm = _t(wl["normal"])[None]
            off = _dot(pts, nrm) - wl["offset"]
            dn = off.abs() - rad
            on = torch.nonzero(dn[:, 0] <= 0)[:, 0]
            key = ("wall", k)
            if key not in self.hist:
                self.hist[key] = torch.zeros_like(pts)
            n = torch.sign(off[on]) * nrm
            c = pts[on] - n * (rad[on] + 0.5 * dn[on]) - self.x[body[on]]
            self.pair_contact(F, M, key, on, dn[on], n, c, None, body[on], None)

    def force(self):
        F = self.g * self.m
        M = torch.zeros_like(F)
        self.contacts(F, M)
        return F, M

    def angular(self, M):
        qi = self.q * torch.tensor([1.0, -1.0, -1.0, -1.0], device=self.q.device, dtype=torch.float64)
        om, mb = _rot(qi, self.s), _rot(qi, M)
        I = self.I
        gy = torch.stack([(I[:, 2] - I[:, 1]) * om[:, 1] * om[:, 2], (I[:, 0] - I[:, 2]) * om[:, 2] * om[:, 0],
                          (I[:, 1] - I[:, 0]) * om[:, 0] * om[:, 1]], 1)
        return _rot(self.q, (mb - gy) / I)

    def first(self):
        """The first force pass leaves the force in place of the acceleration, as the reference's decks do."""
        self.a, _ = self.force()

    def refresh(self):
        F, M = self.force()
        self.a, self.al = F / self.m, self.angular(M)

    def steps(self, k):
        dt = self.w.dt
        for _ in range(k):
            self.x = self.x + self.v * dt + 0.5 * dt * dt * self.a
            self.v = self.v + 0.5 * dt * self.a
            q, s = self.q, self.s
            dq = 0.5 * torch.cat([-_dot(s, q[:, 1:]), _cross(s, q[:, 1:]) + s * q[:, :1]], 1)
            q = q + dt * dq
            self.q = q / _norm(q)
            self.s = s + 0.5 * dt * self.al
            if self.moved():
                self.rebuild()
            self.refresh()
            self.s = self.s + 0.5 * dt * self.al
            self.v = self.v + 0.5 * dt * self.a

    def frame(self):
        return {k: v.t().cpu() for k, v in (("position", self.x + self.wrapped), ("velocity", self.v), ("spin", self.s),
                                            ("orientation", self.q), ("acceleration", self.a))}


class _Spheres(_Exact):
    def __init__(self, w, mesh=None, reach=0.4):
        super().__init__(w)
        i, j = _close_pairs(self.x.clone(), 2.0 * float(self.r.max()) + reach, self.lo, self.hi, self.per)
        sh = self.shifts(i, j)
        gap = (_norm(self.x[i] - self.x[j] - sh) - self.r[i] - self.r[j])[:, 0]
        near = gap < reach
        self.i, self.j, self.sh = i[near], j[near], sh[near]
        listed_ = gap < w.rcut_inc  # the list entries of the build at these positions
        self.li, self.lj, self.lsh = i[listed_], j[listed_], sh[listed_]
        self.hist["pair"] = torch.zeros_like(self.sh)
        if mesh is not None:
            self.mesh_setup(mesh, reach)
        self.relist()

    def gap(self):
        d = self.x[self.i] - self.x[self.j] - self.sh
        dist = _norm(d)
        return d, dist, dist - self.r[self.i] - self.r[self.j]

    def relist(self):
        if self.i is None:
            return
        rv = self.w.rcut_inc
        self.hold["pair"] = (self.gap()[2] < rv)[:, 0]
        self.images("pair", self.i, self.j)
        for name, s, pts, rm in self.mesh or []:
            self.hold[name] = _point_feature(name, self.x[s], pts, self.r[s] + rm + rv, rv)[0]

    def mesh_setup(self, mesh, reach):
        v = _t(mesh["vertices"])
        e = torch.as_tensor(mesh["edges"].astype(np.int64), device=DEV)
        f = torch.as_tensor(mesh["faces"].astype(np.int64), device=DEV)
        self.mesh = []
        near_z = torch.nonzero(((self.x[:, 2] - v[0, 2]).abs() < self.r[:, 0] + reach))[:, 0]
        for name, pts in (("vertex", v[:, None]), ("edge", v[e]), ("face", v[f])):
            lo, hi = pts.amin(1)[:, :2], pts.amax(1)[:, :2]
            got = []
            for part in near_z.split(2048):
                y, r = self.x[part][:, None, :2], self.r[part][:, None] + reach
                at = torch.nonzero(((y > lo - r) & (y < hi + r)).all(-1))
                got.append(torch.stack([part[at[:, 0]], at[:, 1]], 1))
            got = torch.cat(got)
            self.mesh.append((name, got[:, 0], pts[got[:, 1]], mesh["minkowski"]))
            self.hist[("mesh", name)] = torch.zeros((len(got), 3), dtype=torch.float64, device=DEV)

    def contacts(self, F, M):
        d, dist, dn = self.gap()
        on = torch.nonzero((dn[:, 0] < 0) & self.hold["pair"])[:, 0]
        i, j, d, dn = self.i[on], self.j[on], d[on], dn[on]
        n = d / dist[on]
        ci = -n * (self.r[i] + 0.5 * dn)
        self.pair_contact(F, M, "pair", on, dn, n, ci, ci + d, i, j)
        self.walls(F, M, self.x, self.r, torch.arange(len(self.x), device=DEV))
        for name, s, pts, rm in self.mesh or []:
            ok, dn, n = _point_feature(name, self.x[s], pts, self.r[s] + rm)
            on = torch.nonzero(ok & self.hold[name])[:, 0]
            b = s[on]
            c = -n[on] * (self.r[b] + 0.5 * dn[on])
            self.pair_contact(F, M, ("mesh", name), on, dn[on], n[on], c, None, b, None)


def _point_feature(name, x, pts, R, rv=0.0):
    """A point against a vertex, an edge or a planar face (points in order): (contact, dn, unit normal to x). The
    lists' filter is the same test with R enlarged by rv, an edge by rv of its length at both ends."""
    if name == "vertex":
        d = x - pts[:, 0]
        dist = _norm(d)
        return (dist < R)[:, 0], dist - R, d / dist
    if name == "edge":
        a, u = pts[:, 0], pts[:, 1] - pts[:, 0]
        t = _dot(u, x - a) / _dot(u, u)
        d = x - a - t * u
        dist = _norm(d)
        return ((t > -rv) & (t < 1 + rv) & (dist <= R))[:, 0], dist - R, d / dist
    a = pts[:, 0]
    n = _cross(pts[:, 1] - a, pts[:, -1] - a)
    n = n / _norm(n)
    off = _dot(n, x - a)
    inside = torch.ones(len(x), dtype=torch.bool, device=x.device)
    for k in range(pts.shape[1]):
        p, q = pts[:, k], pts[:, (k + 1) % pts.shape[1]]
        inside &= ((_dot(_cross(q - p, x - p), n) > 0) | (_norm(q - p) == 0))[:, 0]
    return inside & (off.abs() <= R)[:, 0], off.abs() - R, torch.sign(off) * n


def _edge_edge(A, B, R):
    Ei, Ej, v = A[:, 1] - A[:, 0], B[:, 1] - B[:, 0], A[:, 0] - B[:, 0]
    c, d, e, g, k = _dot(Ei, Ei), _dot(Ej, Ej), _dot(Ei, Ej), _dot(Ei, v), _dot(Ej, v)
    det = c * d - e * e
    s, t = (e * k - g * d) / det, (c * k - e * g) / det
    n = (A[:, 0] + Ei * s) - (B[:, 0] + Ej * t)
    dist = _norm(n)
    ok = (det.abs() > 1e-12) & (s > 0) & (s < 1) & (t > 0) & (t < 1) & (dist <= R)
    return ok[:, 0], dist - R, n / dist, A[:, 0] + Ei * s


class _Polyhedra(_Exact):
    def __init__(self, w, margin=0.08):
        sh = w.shapes
        self.type = torch.as_tensor(w.particles["type"].astype(np.int64), device=DEV)
        self.sv = _t([[list(s.vertices[k]) for k in range(8)] for s in sh])
        edges = [[tuple(s.edges[k]) if k < s.ne else (0, 0) for k in range(12)] for s in sh]
        # triangles repeat their last vertex, so that every face has four
        faces = [[[s.faces[k][min(a, s.face_size[k] - 1)] if k < s.nf else 0 for a in range(4)] for k in range(8)] for s in sh]
        self.se, self.sf = (torch.as_tensor(v, device=DEV) for v in (edges, faces))
        self.cnt = torch.as_tensor([[s.nv, s.ne, s.nf] for s in sh], device=DEV)
        self.mink = _t([s.minkowski for s in sh])[:, None]
        super().__init__(w)
        self.rm = self.mink[self.type] * self.h
        i, j = _close_pairs(self.x.clone(), 2.0 * float(self.r.max()) + margin, self.lo, self.hi, self.per)
        self.feat, V = {}, self.marks()
        for key, (a, b) in {"vv": (0, 0), "ve": (0, 1), "ev": (1, 0), "vf": (0, 2), "fv": (2, 0), "ee": (1, 1)}.items():
            size = (8, 12, 8)
            got = []
            for lo in range(0, len(i), 1 << 16):
                p, q = i[lo:lo + (1 << 16)], j[lo:lo + (1 << 16)]
                s = self.shifts(p, q)
                pa, pb = self.points(a, V, p, None)[:, :, None], self.points(b, V, q, None)[:, None] + s[:, None, None, None]
                ca, cb = pa.mean(3), pb.mean(3)
                ra = (pa - ca[:, :, :, None]).square().sum(-1).amax(-1).sqrt()
                rb = (pb - cb[:, :, :, None]).square().sum(-1).amax(-1).sqrt()
                lim = (self.rm[p] + self.rm[q])[:, :, None] + margin + ra + rb
                ok = (ca - cb).square().sum(-1).sqrt() < lim
                ok &= torch.arange(size[a], device=DEV)[None, :, None] < self.cnt[self.type[p], a][:, None, None]
                ok &= torch.arange(size[b], device=DEV)[None, None] < self.cnt[self.type[q], b][:, None, None]
                at = torch.nonzero(ok)
                got.append(torch.cat([p[at[:, 0], None], q[at[:, 0], None], at[:, 1:]], 1))
            got = torch.cat(got)
            self.feat[key] = (got, self.shifts(got[:, 0], got[:, 1]), a, b)
            self.hist[key] = torch.zeros((len(got), 3), dtype=torch.float64, device=DEV)
        self.relist()

    def points(self, kind, V, body, sub):
        """The points of the bodies' vertices (0), edges (1) or faces (2): all of them, or one per body."""
        ty = self.type[body]
        if kind == 0:
            idx = torch.arange(8, device=DEV)[None, :, None].expand(len(body), 8, 1)
        else:
            idx = (self.se if kind == 1 else self.sf)[ty]
        if sub is not None:
            idx = idx[torch.arange(len(body), device=DEV), sub]
            return V[body[:, None], idx]
        return V[body[:, None, None], idx]

    def marks(self):
        hv = self.h[:, :, None] * self.sv[self.type]
        return self.x[:, None] + _rot(self.q[:, None], hv)

    def moved(self):
        k = torch.arange(8, device=DEV)[None] < self.cnt[self.type, 0][:, None]
        d = (self.marks() - self.ref).square().sum(-1) * k
        return bool((d >= (0.5 * self.w.rcut_inc) ** 2).any())

    def features(self, key, V, rv=0.0):
        """Test of every candidate of a kind: (flag, dn, normal, point of the vertex side, vertex side, other)."""
        got, sh, a, b = self.feat[key]
        p, q = got[:, 0], got[:, 1]
        A, B = self.points(a, V, p, got[:, 2]), self.points(b, V, q, got[:, 3]) + sh[:, None]
        R = self.rm[p] + self.rm[q] + rv
        if key == "ee":
            return _edge_edge(A, B, R)
        kinds = ("vertex", "edge", "face")
        if a == 0:
            return _point_feature(kinds[b], A[:, 0], B, R, rv) + (A[:, 0],)
        return _point_feature(kinds[a], B[:, 0], A, R, rv) + (B[:, 0],)

    def relist(self):
        if self.feat is not None:
            V = self.marks()
            for key, (got, _, _, _) in self.feat.items():
                self.hold[key] = self.features(key, V, self.w.rcut_inc)[0]
                self.images(key, got[:, 0], got[:, 1])

    def contacts(self, F, M):
        V = self.marks()
        for key, (got, sh, a, b) in self.feat.items():
            ok, dn, n, pt = self.features(key, V)
            on = torch.nonzero(ok & self.hold[key])[:, 0]
            p, q, swap = got[on, 0], got[on, 1], a > 0 and key != "ee"
            cp = pt[on] - n[on] * (self.rm[q if swap else p] + 0.5 * dn[on])
            cpp, cpq = cp - self.x[p], cp - sh[on] - self.x[q]
            if swap:
                self.pair_contact(F, M, key, on, dn[on], n[on], cpq, cpp, q, p, swap=True)
            else:
                self.pair_contact(F, M, key, on, dn[on], n[on], cpp, cpq, p, q)
        k = torch.arange(8, device=DEV)[None] < self.cnt[self.type, 0][:, None]
        body = torch.nonzero(k)
        self.walls(F, M, V[body[:, 0], body[:, 1]], self.rm[body[:, 0]], body[:, 0])


class _Net:
    """The network at 64 bits from unrounded parameters."""

    def __init__(self, params, scales):
        self.sc = scales
        self.flat = torch.as_tensor(np.asarray(params, np.float64), device=DEV)

    def parts(self, flat):
        out, at = {}, 0
        for name, shape in surrogate.param_shapes():
            k = int(np.prod(shape))
            out[name] = flat[at:at + k].reshape(shape)
            at += k
        return out

    def graph(self, e):
        """Node inputs, directed edges and edge inputs at the state of e."""
        sc = self.sc
        i, j = torch.cat([e.li, e.lj]), torch.cat([e.lj, e.li])
        sh = torch.cat([e.lsh, -e.lsh])
        R, w = e.r, e.s
        zero = torch.zeros_like(R)
        x = torch.cat([(R - sc["r0"]) / sc["r0"] * 4.0, w * R / sc["v0"], (R / sc["r0"]) ** 3, zero, zero, zero], 1)
        d = e.x[j] + sh - e.x[i]
        dist = _norm(d)
        n = d / dist
        Rs = R[i] + R[j]
        o = (Rs - dist) / Rs * sc["ov_scale"]
        vr = (e.v[j] - R[j] * _cross(w[j], n) - e.v[i] - R[i] * _cross(w[i], n)) / sc["v0"]
        on = (o > 0).double()
        op = o.clamp(min=0.0)
        vn = on * _dot(vr, n)
        return x, i, j, torch.cat([n, o, vr, (R[j] - R[i]) / Rs * 4.0, op * n, vn * n, op, on], 1)

    def forward(self, graph, flat=None):
        x, i, j, e = graph
        p = self.parts(self.flat if flat is None else flat)
        h = torch.relu(x @ p["W_in"].t() + p["b_in"])
        for l in range(3):
            pq = h @ p[f"W_AB{l}"].t()
            P, Q = pq[:, :128], pq[:, 128:]
            m = torch.zeros_like(h)
            for at in range(0, len(i), 1 << 20):
                a, b = i[at:at + (1 << 20)], j[at:at + (1 << 20)]
                z = P[a] + Q[b] + e[at:at + (1 << 20)] @ p[f"W_E{l}"].t() + p[f"b_E{l}"]
                m = m.index_add(0, a, torch.relu(z))
            h = h + torch.relu(torch.cat([h, 0.125 * m], 1) @ p[f"W_U{l}"].t() + p[f"b_U{l}"])
        return h @ p["W_out"].t() + p["b_out"]


def exact(case, seed):
    kind = case["kind"]
    w = _workload(case, seed)
    if kind.startswith("poly"):
        e = _Polyhedra(w)
    else:
        e = _Spheres(w, mesh=_floor(w) if kind == "mesh" else None)
    e.first()
    if kind not in ("forward", "train", "surrogate"):
        e.steps(case["steps"])
        return e.frame()
    params, scales = surrogate.load(WEIGHTS.get(case["substeps"], surrogate.WEIGHTS))
    K = case["substeps"]
    fs = scales["m0"] * scales["a0"]
    ts = fs * scales["r0"]
    if kind == "forward":
        return _Net(params, scales).forward(_Net(params, scales).graph(e)).cpu()
    e.steps(K)
    T = w.dt * K
    if kind == "train":
        net = _Net(surrogate.init_params(seed), scales)
        graph = net.graph(e)
        v0, s0 = e.v, e.s
        e.steps(K)
        target = torch.cat([e.m * ((e.v - v0) / T - e.g) / fs, e.I * (e.s - s0) / T / ts], 1)
        flat = net.flat.clone().requires_grad_(True)
        loss = (net.forward(graph, flat) - target).square().mean()
        loss.backward()
        # the first Adam update: both moments are those of this gradient
        step = 1e-3 * flat.grad / (flat.grad.abs() + 1e-8)
        return {"loss": float(loss), "used": True, "grads": flat.grad.cpu(), "params": (net.flat - step).cpu()}
    net = _Net(params, scales)
    for _ in range(case["steps"] - 1):
        out = net.forward(net.graph(e))
        a = e.g + fs * out[:, :3] / e.m
        al = ts * out[:, 3:] / e.I
        e.x = e.x + e.v * T + 0.5 * T * T * a
        e.v = e.v + a * T
        q, s = e.q, e.s
        q = q + 0.5 * T * torch.cat([-_dot(s, q[:, 1:]), _cross(s, q[:, 1:]) + s * q[:, :1]], 1)
        e.q = q / _norm(q)
        e.s = s + al * T
    e.refresh()  # the checked window starts from forces at the state the network left
    e.steps(K)
    return e.frame()
