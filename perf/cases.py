"""Performance cases: the solves, right-hand sides and mesh transfers that a
program using this library runs, through its public Python entry points.

A solve starts from fields in hand, advances a number of LSRK4(5) steps on
the device and takes the final state back as host arrays, which is the only
form in which the library hands a state out.  FP32 states come back as
float32, the others as float64.

exact() restates each case in plain torch, in 64 bits, without the library.
"""
import math

import numpy as np
import torch

import bfam_amd as bx
import bfam_amd.workloads as W

PREC = {"fp32": bx.FP32, "fp64": bx.FP64, "fp32_rhs": bx.FP32_RHS}
CUDA = "cuda"


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # an application with its own time integrator: fields in, L(q, t) out.
        # The smallest call; host round trips and launches are what it costs
        {"name": "rhs_n4_N4_fp64", "kind": "rhs", "N": 4, "nx": 4, "ny": 4, "nz": 4,
         "prec": "fp64"},
        # the 2-D acoustic plane-wave configuration: 1,000 tiny launches
        {"name": "acoustic_16x16_N4_fp64", "kind": "acoustic", "N": 4, "nx": 16, "ny": 16,
         "prec": "fp64", "steps": 100},
        # the smallest request the serving loop takes, advanced as it does it
        {"name": "serve_n8_N3_fp32", "kind": "brick", "N": 3, "nx": 8, "ny": 8, "nz": 8,
         "prec": "fp32", "steps": 200, "path": "batch", "bc": False, "forcing": False},
        # requests of the lower orders, single subdomains stepped eagerly:
        # a cube, an odd-sized cube (odd Np), a ragged half space with a free
        # surface and absorbing sides
        {"name": "solve_n30_N3_fp32", "kind": "brick", "N": 3, "nx": 30, "ny": 30, "nz": 30,
         "prec": "fp32", "steps": 300, "path": "step", "bc": False, "forcing": False},
        {"name": "solve_n27_N4_fp32", "kind": "brick", "N": 4, "nx": 27, "ny": 27, "nz": 27,
         "prec": "fp32", "steps": 200, "path": "step", "bc": False, "forcing": False},
        {"name": "halfspace_21x18x25_N5_fp32", "kind": "brick", "N": 5, "nx": 21, "ny": 18,
         "nz": 25, "prec": "fp32", "steps": 200, "path": "step", "bc": True, "forcing": False},
        # the headline configuration (order 7, FP32, captured step replayed)
        # at the size of the largest request and of the precision study
        {"name": "headline_n32_N7_fp32", "kind": "brick", "N": 7, "nx": 32, "ny": 32, "nz": 32,
         "prec": "fp32", "steps": 120, "path": "graph", "bc": False, "forcing": False},
        # the serving loop's default precision, FP32 rates on FP64 state
        {"name": "serve_n17_N6_fp32rhs", "kind": "brick", "N": 6, "nx": 17, "ny": 17, "nz": 17,
         "prec": "fp32_rhs", "steps": 200, "path": "batch", "bc": False, "forcing": False},
        # the precision study's FP64 run: manufactured solution with forcing
        {"name": "mms_n16_N7_fp64", "kind": "brick", "N": 7, "nx": 16, "ny": 16, "nz": 16,
         "prec": "fp64", "steps": 200, "path": "step", "bc": False, "forcing": True},
        # the adapted-mesh configuration: orders 7/5/3 by level, mortar glue
        {"name": "adapted_16_753_fp32", "kind": "octree", "base": 16, "levels": 2,
         "radius": 0.2, "place": 1, "orders": "753", "prec": "fp32", "steps": 200},
        # the serving loop with requests of several orders resident at once
        {"name": "serve_mixed_fp32", "kind": "mixed", "members": "8x7,20x3,11x5,16x4,9x6,13x3",
         "prec": "fp32", "steps": 100},
        # between two steps of an adapted run: the refined sphere has moved
        {"name": "transfer_16_53_fp32", "kind": "transfer", "base": 16, "radius": 0.2,
         "place": 2, "orders": "53", "prec": "fp32"},
    ]


def draw(rng):
    """One more case of the same ranges: bricks of 8 to 32 elements a side
    (ragged), orders 3 to 7, every precision and way of stepping; acoustic
    squares; right-hand sides; adapted meshes; mixed batches; transfers."""
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["brick"] * 6 + ["rhs", "acoustic", "octree", "mixed", "transfer"])
    prec = rng.choice(["fp32", "fp32", "fp32", "fp64", "fp32_rhs"])
    if kind == "acoustic":
        return {"kind": kind, "N": rng.randint(2, 8), "nx": log_int(8, 96), "ny": log_int(8, 96),
                "prec": prec, "steps": log_int(20, 200)}
    if kind == "octree":
        return {"kind": kind, "base": rng.randint(6, 16), "levels": rng.randint(1, 2),
                "radius": round(rng.uniform(0.1, 0.22), 3), "place": rng.randint(1, 99),
                "orders": rng.choice(["753", "643", "654", "543"]), "prec": prec,
                "steps": log_int(20, 150)}
    if kind == "mixed":
        mem = ",".join("%dx%d" % (log_int(6, 18), rng.randint(3, 7))
                       for _ in range(rng.randint(3, 8)))
        return {"kind": kind, "members": mem, "prec": prec, "steps": log_int(10, 100)}
    if kind == "transfer":
        return {"kind": kind, "base": rng.randint(5, 18), "radius": round(rng.uniform(0.1, 0.25), 3),
                "place": rng.randint(1, 99), "orders": rng.choice(["53", "73", "64", "54", "75"]), "prec": prec}
    N = rng.randint(3, 7)
    if kind == "rhs":
        return {"kind": kind, "N": N, "nx": log_int(2, 16), "ny": log_int(2, 16),
                "nz": log_int(2, 16), "prec": prec}
    most = 24 ** 3 * 512 / (1 if prec == "fp32" else 2)
    while True:
        n = [log_int(8, 32) for _ in range(3)]
        if n[0] * n[1] * n[2] * (N + 1) ** 3 <= most:
            break
    return {"kind": "brick", "N": N, "nx": n[0], "ny": n[1], "nz": n[2], "prec": prec,
            "steps": log_int(40, 200), "path": rng.choice(["step", "batch", "graph"]),
            "bc": rng.random() < 0.25, "forcing": rng.random() < 0.15}


# ------------------------------------------------- inputs, from the seed alone

def _dims(case):
    return [case["nx"], case["ny"]] + ([case["nz"]] if "nz" in case else [])


def _spread(bits):
    """Morton keys of integer points (one column per axis)."""
    p = np.asarray(bits, dtype=np.int64)
    key = np.zeros(len(p), dtype=np.int64)
    for b in range(20):
        for d in range(p.shape[1]):
            key |= ((p[:, d] >> b) & 1) << (b * p.shape[1] + d)
    return key


def _points(n):
    """Grid points of a brick in the storage (Morton) order of its elements."""
    g = np.stack(np.meshgrid(*[np.arange(m) for m in n], indexing="ij"), -1).reshape(-1, len(n))
    return g[np.argsort(_spread(g), kind="stable")]


def _lgl(N):
    """Legendre-Gauss-Lobatto nodes and weights."""
    P = np.polynomial.legendre.Legendre.basis(N)
    r = np.concatenate([[-1.0], np.sort(P.deriv().roots().real), [1.0]])
    for _ in range(3):
        d1, d2 = P.deriv()(r[1:-1]), P.deriv(2)(r[1:-1])
        r[1:-1] -= d1 / d2
    r = 0.5 * (r - r[::-1])
    return r, 2.0 / (N * (N + 1) * P(r) ** 2)


def _lagrange(r, y):
    """B[q, i] = l_i(y_q) of the Lagrange basis on the nodes r."""
    n = len(r)
    B = np.ones((len(y), n))
    for i in range(n):
        for k in range(n):
            if k != i:
                B[:, i] *= (np.asarray(y) - r[k]) / (r[i] - r[k])
    return B


def _diff(r):
    n = len(r)
    D = np.zeros((n, n))
    lam = np.array([1 / np.prod([r[j] - r[k] for k in range(n) if k != j]) for j in range(n)])
    for i in range(n):
        for j in range(n):
            if i != j:
                D[i, j] = lam[j] / lam[i] / (r[i] - r[j])
        D[i, i] = -D[i].sum()
    return D


def _material(K, rng):
    """Per-element density and wave speeds, the ranges of the benchmark."""
    rho, cp = rng.uniform(1.5, 3.0, K), rng.uniform(3.0, 6.0, K)
    return rho, cp, cp / rng.uniform(1.6, 2.0, K)


def _fields(x0, h, N, nf, L, rng):
    """Smooth fields of a few wavelengths over the domain, device tensor of
    shape (nf, K, nodes per element)."""
    dim = len(L)
    r = torch.tensor(0.5 * (_lgl(N)[0] + 1), device=CUDA)
    x0, h = torch.tensor(x0, device=CUDA), torch.tensor(h, device=CUDA)
    x = [x0[:, d, None] + h[:, d, None] * r for d in range(dim)]
    shape = [x0.shape[0]] + [N + 1] * dim
    q = torch.zeros([nf] + shape, dtype=torch.float64, device=CUDA)
    for f in range(nf):
        for _ in range(3):
            w = rng.uniform(0.2, 1.0)
            s = [torch.sin(2 * math.pi * int(rng.integers(1, 5)) * x[d] / L[d] +
                           rng.uniform(0, 2 * math.pi)) for d in range(dim)]
            p = w * s[0]
            for d in range(1, dim):
                p = p.unsqueeze(1) * s[d].reshape([shape[0], N + 1] + [1] * d)
            q[f] += p
    return q.reshape(nf, shape[0], -1)


def _source(K, N, h, dt, steps, rng):
    """A Ricker point source at a seeded point of a seeded element."""
    r, w = _lgl(N)
    e, rs = int(rng.integers(K)), rng.uniform(-0.9, 0.9, h.shape[1])
    wt = np.ones(1)
    for d in range(h.shape[1]):
        wt = np.multiply.outer(_lagrange(r, [rs[d]])[0] / (w * 0.5 * h[e, d]), wt)
    T = steps * dt
    return {"elem": e, "weights": np.ascontiguousarray(wt.ravel()),
            "amp": [0, 0, 0, 1, 1, 1, 0, 0, 0] if h.shape[1] == 3 else [1.0, 0, 0],
            "t0": 0.5 * T, "f0": 2.4 / T}


def _dt(hmin, cmax, N):
    return 0.5 * hmin / (cmax * (N + 1) ** 2)


def _brick_inputs(case, seed):
    """Everything about a brick solve that comes from the seed, as numpy
    arrays in storage order, and the initial fields."""
    rng = np.random.default_rng([seed, 1])
    n, N = _dims(case), case["N"]
    dim = len(n)
    hd = np.array([1.0, 1.3, 0.8][:dim]) / max(n)
    L = [hd[d] * n[d] for d in range(dim)]
    pts = _points(n)
    K = len(pts)
    rho, cp, cs = _material(K, rng)
    steps = case.get("steps", 1)
    d = {"n": n, "N": N, "L": L, "pts": pts, "K": K, "h": np.tile(hd, (K, 1)),
         "x0": pts * hd, "rho": rho, "cp": cp, "cs": cs if dim == 3 else None, "steps": steps,
         "bc": bool(case.get("bc")), "dt": _dt(hd.min(), cp.max(), N), "mms": None, "t0": 0.0}
    if case.get("forcing"):
        d["rho"], d["cp"], d["cs"] = np.ones(K), np.full(K, math.sqrt(3.0)), np.ones(K)
        d["dt"] = _dt(hd.min(), math.sqrt(3.0), N)
        d["mms"] = {"k": 2 * math.pi, "omega": 2 * math.pi, "F": rng.uniform(-3, 3, 9)}
    d["src"] = _source(K, N, d["h"], d["dt"], max(steps, 20), rng)
    d["q0"] = _fields(d["x0"], d["h"], N, 9 if dim == 3 else 3, L, rng)
    return d


def _octree_inputs(case):
    """The forest: refined inside a sphere, which then moves a little.  Where
    they are is part of the case, so that its shapes do not depend on the
    seed."""
    rng = np.random.default_rng([case["place"], 2])
    orders = [int(c) for c in case["orders"]][:case.get("levels", 1) + 1]
    return {"base": case["base"], "levels": case.get("levels", 1), "radius": case["radius"],
            "orders": orders, "center": [float(v) for v in rng.uniform(0.35, 0.65, 3)],
            "shift": [float(v) for v in rng.uniform(-0.06, 0.06, 3)]}


# ----------------------------------------------------------------- the library

_device = None


def _dev():
    global _device
    if _device is None:
        _device = bx.Device(0)
    return _device


class _State:
    """Handles of one program: closed when it goes away."""

    def __init__(self, **kw):
        self.subs, self.batch, self.glue = [], None, None
        self.__dict__.update(kw)

    def __del__(self):
        if self.batch is not None:
            self.batch.close()
        if self.glue is not None:
            self.glue.close()
        for s in self.subs:
            s.close()


def _upload(d, precision):
    """A subdomain of a brick, ready to step."""
    dim = len(d["n"])
    mesh = W.Mesh(dim, d["n"], d["N"], L=d["L"], periodic=[0 if d["bc"] else 1] * dim)
    cfg = {"mesh": mesh, "rho": d["rho"], "cp": d["cp"], "cs": d["cs"],
           "physics": bx.ELASTIC3D if dim == 3 else bx.ACOUSTIC2D, "src": d["src"]}
    if d["bc"]:
        cfg["bc"] = W.boundary_kinds(mesh, [bx.BC_ABSORB] * 5 + [bx.BC_FREE])
    if d["mms"]:
        cfg.update(d["mms"])
    return W.upload(_dev(), cfg, precision)


def _host(q):
    return q.reshape(q.shape[0], -1).cpu().numpy()


def prepare(case, seed):
    prec = PREC[case["prec"]]
    kind = case["kind"]
    if kind in ("brick", "acoustic", "rhs"):
        d = _brick_inputs(case, seed)
        sub = _upload(d, prec)
        q0 = _host(d["q0"])
        sub.set_fields(q0, 0.0, d["dt"])
        st = _State(case=case, subs=[sub], q0=q0, dt=d["dt"])
        if case.get("path") in ("batch", "graph"):
            st.batch = bx.Batch(_dev(), st.subs)
        if case.get("path") == "graph":
            st.batch.capture(1)
        return st
    if kind == "mixed":
        st = _State(case=case)
        for d in _members(case, seed):
            sub = _upload(d, prec)
            sub.set_fields(_host(d["q0"]), 0.0, d["dt"])
            st.subs.append(sub)
        st.batch = bx.Batch(_dev(), st.subs)
        return st
    o = _octree_inputs(case)
    if kind == "octree":
        tree = bx.octree(o["base"], o["levels"], o["center"], o["radius"], o["orders"])
        st = _State(case=case)
        _tree_subs(st.subs, tree, seed, prec)
        st.glue = bx.Glue(_dev(), st.subs, tree["mortars"])
        st.batch = bx.Batch(_dev(), st.subs)
        st.batch.set_glue(st.glue)
        st.batch.capture(1)
        return st
    to = [c + s for c, s in zip(o["center"], o["shift"])]
    src = (o["base"], 1, o["center"], o["radius"], o["orders"])
    dst = (o["base"], 1, to, o["radius"], o["orders"])
    st = _State(case=case)
    st.dt = _tree_subs(st.subs, bx.octree(*src), seed, prec)
    st.nsrc = len(st.subs)
    _tree_subs(st.subs, bx.octree(*dst), seed, prec, fields=False)
    st.maps = bx.transfer_maps(dst, src)
    return st


def _members(case, seed):
    return [_brick_inputs({"nx": int(n), "ny": int(n), "nz": int(n), "N": int(N),
                           "steps": case["steps"]}, seed + 1000 * (i + 1))
            for i, (n, N) in enumerate(m.split("x") for m in case["members"].split(","))]


def _tree_subs(out, tree, seed, prec, fields=True):
    """Upload an adapted mesh's subdomains; returns the time step."""
    meshes = [W.SubMesh(s) for s in tree["subs"]]
    mats = [_material(sm.K, np.random.default_rng([seed, 3, sm.N])) for sm in meshes]
    dt = min(_dt(float(sm.h.min()), m[1].max(), sm.N) for sm, m in zip(meshes, mats))
    for sm, (rho, cp, cs) in zip(meshes, mats):
        sub = bx.Subdomain(_dev(), bx.ELASTIC3D, prec, sm.N, sm.r, sm.w, sm.Dr, sm.vmapM,
                           sm.vmapP, sm.h, rho, cp, cs, x0=sm.x0)
        out.append(sub)
        if fields:
            q = _fields(sm.x0, sm.h, sm.N, 9, [1.0] * 3, np.random.default_rng([seed, 4]))
            sub.set_fields(_host(q), 0.0, dt)
    return dt


def _result(subs, prec):
    out = [torch.from_numpy(s.download()) for s in subs]
    return [q.float() for q in out] if prec == "fp32" else out


def run(state):
    case = state.case
    kind = case["kind"]
    if kind == "rhs":
        sub = state.subs[0]
        sub.set_fields(state.q0, 0.0, state.dt)
        r = torch.from_numpy(sub.rhs(0.25 * state.dt))
        return r.float() if case["prec"] != "fp64" else r
    if kind == "transfer":
        src, dst = state.subs[:state.nsrc], state.subs[state.nsrc:]
        bx.transfer_fields(state.maps, src, dst, state.dt)
        return _result(dst, case["prec"])
    steps = case["steps"]
    path = "graph" if kind == "octree" else "batch" if kind == "mixed" else case.get("path", "step")
    if path == "step":
        state.subs[0].step(steps)
    elif path == "batch":  # the serving loop's chunks
        for k in range(0, steps, 10):
            state.batch.step(min(10, steps - k))
    else:
        for _ in range(steps):
            state.batch.launch_graph()
    return _result(state.subs, case["prec"])


def work(case):
    """State in and out of every stage, and the rates' carrier where it is
    read: 11.2 (FP32) or 22.4 bytes per value and stage on average over a
    step, and the result's bytes.  Per value and stage a derivative of
    2 (N+1) flops for each of the axes it feeds (18 over nine fields; four
    over three in 2-D), and about 17 for the rest."""
    kind = case["kind"]
    if kind in ("brick", "rhs", "acoustic"):
        n = _dims(case)
        parts = [(case["N"], math.prod(n), len(n))]
    elif kind == "mixed":
        parts = [(int(N), int(n) ** 3, 3) for n, N in
                 (m.split("x") for m in case["members"].split(","))]
    else:
        o = _octree_inputs(case)
        parts = [(N, len(p), 3) for N, p in zip(o["orders"], _leaves(o, o["center"]))]
    size = 4 if case["prec"] == "fp32" else 8
    stages = 5 * case.get("steps", 0)
    b = f = 0.0
    for N, K, dim in parts:
        nf = 9 if dim == 3 else 3
        dof = nf * K * (N + 1) ** dim
        deriv = 4 * (N + 1) if dim == 3 else 8 * (N + 1) / 3
        b += dof * (stages * (11.2 if size == 4 else 22.4) + size)
        f += dof * stages * (deriv + 17)
        if kind == "rhs":
            b, f = b + 8 * dof + size * dof, f + dof * (deriv + 12)
        if kind == "transfer":  # three 1-D passes, in 64 bits
            b, f = b + size * dof, f + dof * 6 * (N + 1)
    return {"bytes": b, "flops": f}


# ------------------------------------------- the same in 64 bits, plain torch

KC_A = [0.0, -567301805773 / 1357537059087, -2404267990393 / 2016746695238,
        -3550918686646 / 2091501179385, -1275806237668 / 842570457699]
KC_B = [1432997174477 / 9575080441755, 5161836677717 / 13612068292357,
        1720146321549 / 2090206949498, 3134564353537 / 4481467310338,
        2277821191437 / 14882151754819]
KC_C = [0.0, 1432997174477 / 9575080441755, 2526269341429 / 6820363962896,
        2006345519317 / 3224310063776, 2802321613138 / 2924317926251]
# stress entry of (component, axis) among s11 s22 s33 s12 s13 s23
STRESS = [[3, 6, 7], [6, 4, 8], [7, 8, 5]]


def _t(a, dtype=torch.float64):
    return torch.tensor(np.ascontiguousarray(a), dtype=dtype, device=CUDA)


class _Plain:
    """Elements of one order: fields (nf, K, nodes...), the axes of the nodes
    slowest first (k, j, i), in 64 bits."""

    def __init__(self, N, h, rho, cp, cs, q0, nb, kind=None):
        self.N, self.dim, self.K = N, h.shape[1], len(rho)
        self.nf = 9 if self.dim == 3 else 3
        r, w = _lgl(N)
        self.D, self.w = _t(_diff(r)), w
        self.shape = [self.K] + [N + 1] * self.dim
        self.q = q0.to(torch.float64).reshape([self.nf] + self.shape).clone()
        self.dq = torch.zeros_like(self.q)
        col = [self.K] + [1] * self.dim
        self.g = [_t(2 / h[:, d]).reshape(col) for d in range(self.dim)]
        cs = np.zeros_like(cp) if cs is None else cs
        self.Zp, self.Zs = _t(rho * cp), _t(rho * cs)
        self.rhoi = _t(1 / rho).reshape(col)
        self.lam, self.mu = _t(rho * (cp ** 2 - 2 * cs ** 2)).reshape(col), _t(rho * cs ** 2).reshape(col)
        self.nb = [_t(x, torch.int64) for x in nb]  # own index: a boundary or glued face
        self.kind = kind  # per face: None, or boundary kinds (all its faces alike)
        self.src = self.mms = None

    def face(self, q, f):
        """The trace on face f, last axis the faster tangential one."""
        return q.select(q.dim() - 1 - f // 2, self.N if f & 1 else 0)

    def names(self, A):
        """velocity and traction fields of a face normal to axis A"""
        if self.dim == 2:
            return [1 + A], [0]
        return [0, 1, 2], [STRESS[c][A] for c in range(3)]

    def trace(self, f):
        v, s = self.names(f // 2)
        return [self.face(self.q[c], f) for c in v + s]

    def fluct(self, f, um, up, Zpm, Zsm, Zpp, Zsp):
        """Exact-Riemann fluctuations of velocity and traction on face f."""
        A, s = f // 2, 1.0 if f & 1 else -1.0
        if self.dim == 2:
            return [(Zpp * s * (up[0] - um[0]) + (um[1] - up[1])) / (Zpm + Zpp)]
        dv, dT = [None] * 3, [None] * 3
        den = Zsm + Zsp
        inv = torch.where(den > 0, 1 / torch.where(den > 0, den, 1.0), 0.0)
        for c in range(3):
            jv, jS = up[c] - um[c], up[3 + c] - um[3 + c]
            if c == A:
                d = (Zpp * s * jv + jS) / (Zpm + Zpp)
                dv[c], dT[c] = s * d, s * Zpm * d
            else:
                d = (Zsp * jv + s * jS) * inv
                dv[c], dT[c] = d, Zsm * d
        return dv + dT

    def face_values(self, f):
        um, nb = self.trace(f), self.nb[f]
        col = [self.K] + [1] * (self.dim - 1)
        up = [u[nb] for u in self.trace(f ^ 1)]
        if self.kind:
            edge = (nb == torch.arange(self.K, device=CUDA)).reshape(col)
            half = len(um) // 2 if self.dim == 3 else 1
            free = self.kind[f] == bx.BC_FREE  # else absorbing
            up = [torch.where(edge, (u if (c < half) else -u) if free else 0 * u, x)
                  for c, (u, x) in enumerate(zip(um, up))]
        Z = [z.reshape(col) for z in (self.Zp, self.Zs, self.Zp[nb], self.Zs[nb])]
        return self.fluct(f, um, up, *Z)

    def deriv(self, u, A):
        n, K = self.N + 1, self.K
        if A == 0:
            d = u.reshape(-1, n) @ self.D.T
        elif A == 1:
            d = self.D @ u.reshape(-1, n, n)
        else:
            d = self.D @ u.reshape(K, n, n * n)
        return d.reshape(self.shape) * self.g[A]

    def rates(self, t, glued=None):
        R = torch.zeros_like(self.q)
        for A in range(self.dim):
            v, s = self.names(A)
            if self.dim == 2:
                R[0] -= self.lam * self.deriv(self.q[1 + A], A)
                R[1 + A] -= self.rhoi * self.deriv(self.q[0], A)
            else:
                self.add(R, A, [self.deriv(self.q[c], A) for c in v + s])
        for f in range(2 * self.dim):
            A, s = f // 2, 1.0 if f & 1 else -1.0
            val = self.face_values(f)
            if glued:
                for e, x in glued.get(f, []):
                    val = [u.index_copy(0, e, y) for u, y in zip(val, x)]
            at = [slice(None)] * (1 + self.dim)
            at[self.dim - A] = self.N if f & 1 else 0
            lift = (self.g[A] / self.w[0]).flatten().reshape([self.K] + [1] * (self.dim - 1))
            if self.dim == 2:
                one = [self.K, 1]
                R[1 + A][tuple(at)] += s * lift * self.Zp.reshape(one) * self.rhoi.reshape(one) * val[0]
                R[0][tuple(at)] -= lift * self.lam.reshape(one) * val[0]
            else:
                # s dv enters the stresses as a normal derivative does
                self.add(R, A, [s * lift * x for x in val[:3]] + [lift * x for x in val[3:]], at)
        if self.src:
            x = math.pi * self.src["f0"] * (t - self.src["t0"])
            g = (1 - 2 * x * x) * math.exp(-x * x)
            w = _t(self.src["weights"]).reshape(self.shape[1:])
            for c, a in enumerate(self.src["amp"][:self.nf]):
                R[c, self.src["elem"]] += a * g * w
        if self.mms:
            for c in range(9):
                T = math.sin if c < 3 else math.cos
                R[c] += self.mms["F"][c] * T(self.mms["omega"] * t) * self.pattern(c)
        return R

    def add(self, R, A, d, at=None):
        """Fold derivatives (or lifted fluctuations) along axis A of the three
        velocities and of the traction column into the rates."""
        i = tuple(at) if at is not None else slice(None)
        flat = (lambda x: x) if at is None else (lambda x: x.reshape([self.K, 1, 1]))
        rhoi, lam, mu = flat(self.rhoi), flat(self.lam), flat(self.mu)
        for c in range(3):
            R[c][i] += rhoi * d[3 + c]
            R[3 + c][i] += (lam + 2 * mu if c == A else lam) * d[A]
            if c != A:
                R[STRESS[c][A]][i] += mu * d[c]

    def pattern(self, c):
        x = self.mms["x"]
        S, C = [torch.sin(self.mms["k"] * v) for v in x], [torch.cos(self.mms["k"] * v) for v in x]
        s = {0: (0,), 1: (1,), 2: (2,), 6: (0, 1), 7: (0, 2), 8: (1, 2)}.get(c, ())
        p = [S[d] if d in s else C[d] for d in range(3)]
        return p[0] * p[1] * p[2]

    def update(self, R, k, dt):
        self.dq.mul_(KC_A[k]).add_(R, alpha=dt)
        self.q.add_(self.dq, alpha=KC_B[k])


def _brick_plain(d):
    n, pts = d["n"], d["pts"]
    dim = len(n)
    at = np.full(n, 0)
    at[tuple(pts.T)] = np.arange(len(pts))
    nb = []
    for f in range(2 * dim):
        p = pts.copy()
        p[:, f // 2] += 1 if f & 1 else -1
        out = (p[:, f // 2] < 0) | (p[:, f // 2] >= n[f // 2])
        x = at[tuple((p % n).T)]
        nb.append(np.where(out, np.arange(len(pts)), x) if d["bc"] else x)
    kind = [bx.BC_ABSORB] * 5 + [bx.BC_FREE] if d["bc"] else None
    P = _Plain(d["N"], d["h"], d["rho"], d["cp"], d["cs"], d["q0"], nb, kind)
    P.src = d["src"]
    if d["mms"]:
        r = _lgl(d["N"])[0]
        P.mms = dict(d["mms"], x=[])
        for a in range(3):
            x = _t(d["x0"][:, a, None] + 0.5 * (r + 1) * d["h"][:, a, None])
            s = [len(pts), 1, 1, 1]
            s[3 - a] = d["N"] + 1
            P.mms["x"].append(x.reshape(s))
    return P


def _march(parts, dt, steps, glue=None):
    t = 0.0
    for _ in range(steps):
        for k in range(5):
            extra = glue() if glue else [None] * len(parts)
            R = [p.rates(t + KC_C[k] * dt, x) for p, x in zip(parts, extra)]
            for p, r in zip(parts, R):
                p.update(r, k, dt)
        t += dt
    return [p.q.reshape(p.nf, -1) for p in parts]


def _leaves(o, center):
    """Anchors (in units of their own level's grid) of the leaves of each
    level, Morton order: trees meeting the sphere refined level by level,
    then refined until faces are 2:1."""
    B, L = o["base"], o["levels"]
    F = B << L
    leaf = [set() for _ in range(L + 1)]
    leaf[0] = {(x, y, z) for x in range(B) for y in range(B) for z in range(B)}

    def split(l, p):
        leaf[l].discard(p)
        leaf[l + 1].update((2 * p[0] + (c & 1), 2 * p[1] + (c >> 1 & 1), 2 * p[2] + (c >> 2))
                           for c in range(8))

    for l in range(L):
        s = (1 << (L - l)) / F
        for p in list(leaf[l]):
            e = [max((p[d] << (L - l)) / F - center[d], center[d] - ((p[d] << (L - l)) / F + s), 0.0)
                 for d in range(3)]
            if e[0] * e[0] + e[1] * e[1] + e[2] * e[2] <= o["radius"] ** 2:
                split(l, p)
    again = True
    while again:
        again = False
        for l in range(2, L + 1):
            for p in list(leaf[l]):
                for f in range(6):
                    c = list(p)
                    c[f // 2] = (c[f // 2] + (1 if f & 1 else -1)) % (B << l)
                    for m in range(l - 1):
                        b = tuple(v >> (l - m) for v in c)
                        if b in leaf[m]:
                            split(m, b)
                            again = True
    out = []
    for s in leaf:
        p = np.array(sorted(s), dtype=np.int64).reshape(-1, 3)
        out.append(p[np.argsort(_spread(p), kind="stable")])
    return out


def _mass(r):
    """Exact mass matrix of the Lagrange basis on r."""
    x, w = np.polynomial.legendre.leggauss(len(r))
    B = _lagrange(r, x)
    return B.T @ (w[:, None] * B)


def _faces2(a, b, u):
    """The operators a and b along the faster and slower axis of faces u."""
    return torch.einsum("ij,eqj->eqi", a, torch.einsum("pq,eqj->epj", b, u))


def _glue_plain(o, leaves, parts):
    """The hanging faces of an adapted mesh, as a function giving, for each
    order, the fluctuations of its glued faces from both traces on the
    quarter faces of the order of the finer space."""
    B = o["base"]
    where = [{tuple(p): i for i, p in enumerate(lv)} for lv in leaves]
    jobs = []
    for l in range(len(leaves) - 1):
        for f in range(6):
            A = f // 2
            t1, t2 = [d for d in range(3) if d != A]
            quads = [[], [], [], []]
            for i, p in enumerate(leaves[l]):
                c = [int(v) for v in p]
                c[A] = (c[A] + (1 if f & 1 else -1)) % (B << l)
                c = [2 * v for v in c]
                c[A] += 0 if f & 1 else 1
                if tuple(c) not in where[l + 1]:
                    continue
                for q in range(4):
                    s = list(c)
                    s[t1] += q & 1
                    s[t2] += q >> 1
                    quads[q].append((i, where[l + 1][tuple(s)]))
            if quads[0]:
                jobs.append((l, f, [_t(np.array(x), torch.int64) for x in quads]))
    ops = {}
    for l in range(len(leaves) - 1):
        Nb, Ns = o["orders"][l], o["orders"][l + 1]
        rg = _lgl(max(Nb, Ns))[0]
        (rb, wb), (rs, ws) = _lgl(Nb), _lgl(Ns)
        M = _mass(rg)
        up = [_lagrange(rb, 0.5 * (rg + s)) for s in (-1, 1)]
        Is = _lagrange(rs, rg)
        ops[l] = ([_t(x) for x in up], _t(Is), [_t(x.T @ (0.5 * M) / wb[:, None]) for x in up],
                  _t(Is.T @ M / ws[:, None]))

    def glue():
        out = [{} for _ in leaves]
        for l, f, quads in jobs:
            up, Is, back, Ws = ops[l]
            b, s = parts[l], parts[l + 1]
            tb, ts = b.trace(f), s.trace(f ^ 1)
            total = None
            for q in range(4):
                eb, es = quads[q][:, 0], quads[q][:, 1]
                ub = [_faces2(up[q & 1], up[q >> 1], u[eb]) for u in tb]
                us = [_faces2(Is, Is, u[es]) for u in ts]
                Z = [z.reshape(-1, 1, 1) for z in (b.Zp[eb], b.Zs[eb], s.Zp[es], s.Zs[es])]
                vb = b.fluct(f, ub, us, *Z)
                vs = s.fluct(f ^ 1, us, ub, Z[2], Z[3], Z[0], Z[1])
                vb = [_faces2(back[q & 1], back[q >> 1], v) for v in vb]
                total = vb if total is None else [x + y for x, y in zip(total, vb)]
                out[l + 1].setdefault(f ^ 1, []).append((es, [_faces2(Ws, Ws, v) for v in vs]))
            out[l].setdefault(f, []).append((quads[0][:, 0], total))
        return out

    return glue


def _tree_plain(o, leaves, seed):
    parts = []
    for l, p in enumerate(leaves):
        n, N = o["base"] << l, o["orders"][l]
        h = np.full((len(p), 3), 1.0 / n)
        rho, cp, cs = _material(len(p), np.random.default_rng([seed, 3, N]))
        at = {tuple(x): i for i, x in enumerate(p)}
        nb = []
        for f in range(6):
            c = p.copy()
            c[:, f // 2] = (c[:, f // 2] + (1 if f & 1 else -1)) % n
            nb.append(np.array([at.get(tuple(x), i) for i, x in enumerate(c)]))
        q0 = _fields(p / n, h, N, 9, [1.0] * 3, np.random.default_rng([seed, 4]))
        parts.append(_Plain(N, h, rho, cp, cs, q0, nb))
        parts[-1].dt = _dt(1.0 / n, cp.max(), N)
    return parts


def _transfer_plain(o, seed):
    """Fields of one refined mesh on the other: kept, interpolated onto
    children, or the L2 projection of eight children."""
    to = [c + s for c, s in zip(o["center"], o["shift"])]
    old, new = _leaves(o, o["center"]), _leaves(o, to)
    where = [{tuple(p): i for i, p in enumerate(lv)} for lv in old]
    q = [_fields(p / (o["base"] << l), np.full((len(p), 3), 1.0 / (o["base"] << l)), N, 9,
                 [1.0] * 3, np.random.default_rng([seed, 4]))
         for l, (p, N) in enumerate(zip(old, o["orders"]))]
    N0, N1 = o["orders"]
    rg, r0, r1 = (_lgl(n)[0] for n in (max(N0, N1), N0, N1))
    M = _mass(rg)
    down = np.linalg.solve(_mass(r1), _lagrange(r1, rg).T @ M)  # glue grid -> children's order
    fine = [_t(down @ _lagrange(r0, 0.5 * (rg + s))) for s in (-1, 1)]
    coarse = [_t(np.linalg.solve(_mass(r0), _lagrange(r0, 0.5 * (rg + s)).T @ (0.5 * M))
                 @ _lagrange(r1, rg)) for s in (-1, 1)]

    def apply(ops, c, u, n):
        u = u.reshape(9, -1, n + 1, n + 1, n + 1)
        return torch.einsum("ai,bj,ck,fekji->fecba", ops[c & 1], ops[c >> 1 & 1], ops[c >> 2], u)

    out = [torch.zeros(9, len(p), (n + 1) ** 3, dtype=torch.float64, device=CUDA)
           for p, n in zip(new, o["orders"])]
    for l, p in enumerate(new):
        keep = [(i, where[l][tuple(x)]) for i, x in enumerate(p) if tuple(x) in where[l]]
        a, b = _t(np.array(keep), torch.int64).T
        out[l][:, a] = q[l][:, b]
    for c in range(8):
        bit = [c & 1, c >> 1 & 1, c >> 2]
        born = [(i, where[0][tuple(x // 2)]) for i, x in enumerate(new[1])
                if tuple(x) not in where[1] and list(x % 2) == bit]
        if born:
            a, b = _t(np.array(born), torch.int64).T
            out[1][:, a] = apply(fine, c, q[0][:, b], N0).reshape(9, len(born), -1)
        gone = [(i, where[1][tuple(2 * x + bit)]) for i, x in enumerate(new[0])
                if tuple(x) not in where[0]]
        if gone:
            a, b = _t(np.array(gone), torch.int64).T
            out[0][:, a] += apply(coarse, c, q[1][:, b], N1).reshape(9, len(gone), -1)
    return [x.reshape(9, -1) for x in out]


def exact(case, seed):
    kind = case["kind"]
    if kind in ("brick", "acoustic"):
        d = _brick_inputs(case, seed)
        return [q.cpu() for q in _march([_brick_plain(d)], d["dt"], d["steps"])]
    if kind == "rhs":
        d = _brick_inputs(case, seed)
        P = _brick_plain(d)
        return P.rates(0.25 * d["dt"]).reshape(P.nf, -1).cpu()
    if kind == "mixed":
        return [_march([_brick_plain(d)], d["dt"], d["steps"])[0].cpu()
                for d in _members(case, seed)]
    o = _octree_inputs(case)
    # the library numbers an adapted mesh's subdomains by increasing order
    by_order = np.argsort(o["orders"], kind="stable")
    if kind == "transfer":
        out = _transfer_plain(o, seed)
    else:
        leaves = _leaves(o, o["center"])
        parts = _tree_plain(o, leaves, seed)
        out = _march(parts, min(p.dt for p in parts), case["steps"], _glue_plain(o, leaves, parts))
    return [out[i].cpu() for i in by_order]
