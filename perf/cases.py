"""The workloads the framework's speed is measured on: time steps of the solvers a PFEM program
runs, through the package's public classes, from the smallest meshes (launch latency) to the
largest ones that fill the GPU.

A pass restarts from the initial node states and positions, advances the case by its steps and
reads the node states and positions back, as a program does between two output times; the solver's
handle, the mesh on the device and the step workspace are made in ``prepare``, except in the
"newmesh" cases, where taking over the mesher's new triangulation is part of the pass, as it is
after every remesh.

``exact`` restates each step in plain torch (FP64, element by element from the P1 formulas, linear
systems solved to 1e-12 or better)."""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

import pfem_amd
from pfem_amd import meshgen as mg

K0, K0P, RHO0 = 2.2e9, 7.0, 1000.0
WC_SC, WC_MAXDT = 0.5, 1e-3
HEAT_MAT = dict(rho=8000.0, cv=500.0, k=50.0)
BQ_MAT = dict(rho=1000.0, mu=1e-2, cv=4000.0, k=50.0, alpha=2e-3, Tr=330.0)


def listed():
    return [
        # the reference's own CPU-sized 2D dam break: a short run of a small case, FP64
        dict(name="pspg2d_dambreak_1k", family="pspg", dim=2, mesh="dambreak", nodes=1001, precision="fp64", rtol=1e-12,
             dt=1e-3, steps=3),
        # an everyday 2D incompressible step (multigrid), FP64
        dict(name="pspg2d_column_20k", family="pspg", dim=2, mesh="column", nodes=20000, precision="fp64", rtol=1e-10,
             dt=1e-3, steps=1),
        # the same in 3D below the multigrid's size, FP64
        dict(name="pspg3d_column_12k", family="pspg", dim=3, mesh="column", nodes=12000, precision="fp64", rtol=1e-10,
             dt=5e-4, steps=1),
        # a production 3D dam break, FP64 multigrid
        dict(name="pspg3d_dambreak_263k", family="pspg", dim=3, mesh="dambreak", nodes=262701, precision="fp64",
             rtol=1e-10, dt=5e-4, steps=1),
        # FP32 inner solves inside FP64 refinement on a ragged 3D column field
        dict(name="pspg3d_field_mixed_ir", family="pspg", dim=3, mesh="field", nodes=72000, precision="mixed_ir",
             rtol=1e-10, dt=5e-4, steps=1),
        # the step after a remesh: a Delaunay mesh taken over from the mesher, then one step
        dict(name="newmesh3d_50k", family="newmesh", dim=3, nodes=50000, rtol=1e-10, dt=5e-4),
        # continuous batching of many independent cases, mixed precision / FP32 state
        dict(name="serving_mixed_40", family="serving", requests=40, lo=2000, hi=60000, rtol=1e-8),
        # weakly compressible: a small 2D tank over many steps (latency), FP64 state
        dict(name="wc2d_tank_2k", family="wc", dim=2, nodes=2000, state="fp64", steps=100),
        # an ordinary 3D tank, FP64 state
        dict(name="wc3d_tank_100k", family="wc", dim=3, nodes=100000, state="fp64", steps=100),
        # the 2.06M-node sloshing tank, FP32 state
        dict(name="wc3d_tank_2m_fp32", family="wc", dim=3, nodes=2060451, state="fp32", steps=100),
        # heat conduction in a block
        dict(name="heat3d_69k", family="heat", dim=3, n=40, steps=10),
        # the fractional-step solver in a lid-driven cavity
        dict(name="frac3d_16k", family="frac", dim=3, n=24, steps=1),
    ]


def draw(rng):
    """A case of the listed ones' ranges."""
    def lognodes(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["pspg2", "pspg2", "pspg3", "pspg3", "ir", "newmesh", "serving", "wc2", "wc3", "wc3", "heat", "frac"])
    if kind == "pspg2":
        return dict(family="pspg", dim=2, mesh="column", nodes=lognodes(500, 60000),
                    precision=rng.choice(["fp64", "fp64", "mixed"]), rtol=1e-10, dt=1e-3, steps=1)
    if kind == "pspg3":
        return dict(family="pspg", dim=3, mesh="column", nodes=lognodes(1000, 200000),
                    precision=rng.choice(["fp64", "fp64", "mixed"]), rtol=1e-10, dt=5e-4, steps=1)
    if kind == "ir":
        return dict(family="pspg", dim=3, mesh="field", nodes=lognodes(3000, 72000), precision="mixed_ir", rtol=1e-10,
                    dt=5e-4, steps=1)
    if kind == "newmesh":
        dim = rng.choice([2, 3])
        return dict(family="newmesh", dim=dim, nodes=lognodes(2000, 50000), rtol=1e-10, dt=1e-3 if dim == 2 else 5e-4)
    if kind == "serving":
        return dict(family="serving", requests=rng.randint(8, 40), lo=2000, hi=lognodes(10000, 60000), rtol=1e-8)
    if kind in ("wc2", "wc3"):
        dim = 2 if kind == "wc2" else 3
        return dict(family="wc", dim=dim, nodes=lognodes(800, 1000000), state=rng.choice(["fp64", "fp32"]),
                    steps=rng.randint(40, 100))
    if kind == "heat":
        dim = rng.choice([2, 3])
        return dict(family="heat", dim=dim, n=lognodes(30, 300) if dim == 2 else rng.randint(8, 48), steps=rng.randint(2, 10))
    dim = rng.choice([2, 3])
    return dict(family="frac", dim=dim, n=rng.randint(16, 60) if dim == 2 else rng.randint(6, 24), steps=1)


# ------------------------------------------------------------------------------------------
# inputs
# ------------------------------------------------------------------------------------------
@functools.lru_cache(maxsize=1)
def _context():
    return pfem_amd.Context(0)


@functools.lru_cache(maxsize=4)
def _lattice(kind, dim, size):
    """The mesh of one size; every seed jitters its interior nodes anew."""
    if kind == "dambreak":
        # 2D: 1.0 x 2.0 m column in a 4 x 3 m tank; 3D: 0.5 x 0.5 x 1.0 m column, h from the node count
        if dim == 2:
            return mg.dambreak_2d(h=0.05 * math.sqrt(1001 / size))
        return mg.dambreak_3d(h=0.01 * (262701 / size) ** (1 / 3))
    if kind == "column":
        return (mg.column_2d_nodes if dim == 2 else mg.column_3d_nodes)(size)
    if kind == "field":
        n = max(4, int(round(size ** (1 / 3))) - 1)
        return mg.randomwalk_3d(ncol=n, mean_cells=n)
    if kind == "tank":
        return mg.tank_3d() if size == 2060451 else mg.tank_nodes(dim, size)
    return mg.cavity(dim, size)


def _mesh(kind, dim, size, seed):
    base = _lattice(kind, dim, size)
    rng = np.random.default_rng(seed)
    pos = np.round(base.pos / base.h) * base.h
    moving = (base.flags & mg.BOUND) == 0
    pos[:, moving] += rng.uniform(-0.1, 0.1, (dim, int(moving.sum()))) * base.h
    return mg.PfemMesh(dim, pos, base.conn, base.flags, base.h, surface=base.surface, meta=base.meta)


def _pspg_state(m, seed):
    """The hydrostatic column with a small seeded motion, still on the walls."""
    q = mg.pspg_hydrostatic(m)
    rng = np.random.default_rng(seed + 1)
    c = rng.uniform(-0.05, 0.05, (m.dim, m.dim + 1))
    L = m.pos.max(axis=1, keepdims=True)
    s = m.pos / np.where(L > 0, L, 1.0)
    v = c[:, :1] + c[:, 1:] @ s
    v[:, (m.flags & mg.BOUND) != 0] = 0.0
    q[:m.dim * m.n_nodes] = v.reshape(-1)
    return q


def _wc_state(m, seed):
    rng = np.random.default_rng(seed + 1)
    v, p, rho, a = mg.wc_tait_hydrostatic(m, K0=K0, K0p=K0P, rho_star=RHO0, u0=float(rng.uniform(0.05, 0.15)))
    return np.concatenate([v.reshape(-1), p, rho, a.reshape(-1)])


def _pspg_case(dim, precision, rtol):
    kw = dict(rho=1000.0, mu=1e-3, residual="Ax_f", min_res=1e-6, max_iter=10, precision=precision, krylov_rtol=rtol,
              krylov_max_iter=40000)
    if precision == "mixed_ir":
        kw.update(precond="jacobi", inner_rtol=3e-2, inner_max_iter=200)
    return pfem_amd.MomContEqIncompNewton(_context(), dim, **kw)


def _wc_case(dim, state):
    return pfem_amd.WCompNewtonStep(_context(), dim, mu=1e-3, K0=K0, K0p=K0P, rho_star=RHO0, wc_state=state)


def _serving_requests(case, seed):
    """The requests of a stream: 60 % 2D, half incompressible columns, half compressible tanks; the
    sizes belong to the case, the jitter and the initial motion to the seed."""
    rng = np.random.default_rng([case["requests"], case["lo"], case["hi"]])
    out = []
    for i in range(case["requests"]):
        dim = 2 if rng.random() < 0.6 else 3
        size = int(math.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"]))))
        kind = "PSPG" if (i % 2 == 0) else "WC"
        m = (mg.column_2d_nodes if dim == 2 else mg.column_3d_nodes)(size, seed=seed * 1000 + i) if kind == "PSPG" \
            else mg.tank_nodes(dim, size, seed=seed * 1000 + i)
        q = _pspg_state(m, seed * 1000 + i) if kind == "PSPG" else _wc_state(m, seed * 1000 + i)
        out.append(dict(kind=kind, mesh=m, q=q))
    return out


def _heat_inputs(case, seed):
    """A block between a hot floor and a cold ceiling, insulated sides, a disturbed temperature."""
    m = _mesh("cavity", case["dim"], case["n"], seed)
    top, bottom = m.meta["top"], m.meta["bottom"]
    fl = np.where(top | bottom, mg.DIRICHLET | mg.FIXED, mg.FIXED).astype(np.uint8)
    hm = mg.PfemMesh(m.dim, m.pos, m.conn, fl, m.h)
    rng = np.random.default_rng(seed + 1)
    Tbc = np.where(bottom, 360.0, np.where(top, 300.0, 0.0))
    T0 = np.where(bottom, 360.0, np.where(top, 300.0, 330.0 + rng.normal(scale=2.0, size=m.n_nodes)))
    return hm, T0, Tbc, 0.5


def _frac_inputs(case, seed):
    m = _mesh("cavity", case["dim"], case["n"], seed)
    rng = np.random.default_rng(seed + 1)
    vbc = np.zeros((m.dim, m.n_nodes))
    vbc[0, m.meta["lid"]] = rng.uniform(0.8, 1.2)
    return m, np.concatenate([vbc.reshape(-1), np.zeros(m.n_nodes)]), vbc, 1e-3


def _frac_kw(dim):
    return dict(rho=1000.0, mu=1e-2, body_force=[0.0] * (dim - 1) + [-9.81], gammaFS=1.0, residual="U", min_res=1e-6,
                max_iter=10)


def _newmesh_cloud(case, seed):
    """The dam-break column's nodes as a remesh finds them, triangulated by the mesher."""
    m = _mesh("column", case["dim"], case["nodes"], seed)
    q = _pspg_state(m, seed)
    t = pfem_amd.Mesher(case["dim"], hchar=m.h, alpha=1.2, omega=0.7, gamma=0.35, addOnFS=True)
    t.set_nodes(m.pos, m.flags, q.reshape(case["dim"] + 1, -1))
    t.triangulate()
    return t


def prepare(case, seed):
    f, dim = case["family"], case.get("dim")
    if f == "pspg":
        m = _mesh(case["mesh"], dim, case["nodes"], seed)
        c = _pspg_case(dim, case["precision"], case["rtol"])
        c.set_mesh(m)
        c.reserve_workspace()
        return dict(case=case, c=c, q=_pspg_state(m, seed), pos=m.pos)
    if f == "newmesh":
        return dict(case=case, c=_pspg_case(dim, "fp64", case["rtol"]), mesher=_newmesh_cloud(case, seed))
    if f == "serving":
        reqs = _serving_requests(case, seed)
        for r in reqs:
            d = r["mesh"].dim
            r["c"] = _pspg_case(d, "mixed", case["rtol"]) if r["kind"] == "PSPG" else _wc_case(d, "fp32")
            r["c"].set_mesh(r["mesh"])
            r["dt"] = 1e-3 if d == 2 else 5e-4
            if r["kind"] == "WC":
                r["c"].set_state(r["q"])
                r["dt"] = r["c"].computeNextDT(WC_SC, WC_MAXDT)
        srv = pfem_amd.Server(_context(), hbm_budget=24 << 30, max_inflight=64, wc_security_coeff=WC_SC,
                              wc_max_dt=WC_MAXDT)
        return dict(case=case, reqs=reqs, srv=srv)
    if f == "wc":
        m = _mesh("tank", dim, case["nodes"], seed)
        c = _wc_case(dim, case["state"])
        c.set_mesh(m)
        return dict(case=case, c=c, q=_wc_state(m, seed), pos=m.pos)
    if f == "heat":
        m, T0, Tbc, dt = _heat_inputs(case, seed)
        c = pfem_amd.HeatEqIncompNewton(_context(), dim, krylov_rtol=1e-10, **HEAT_MAT)
        c.set_mesh(m)
        c.set_dirichlet_T(Tbc)
        return dict(case=case, c=c, q=T0, dt=dt)
    m, q, vbc, dt = _frac_inputs(case, seed)
    c = pfem_amd.MomContEqFracStep(_context(), dim, krylov_rtol=1e-10, **_frac_kw(dim))
    c.set_mesh(m)
    c.set_dirichlet(vbc)
    return dict(case=case, c=c, q=q, pos=m.pos, dt=dt)


# ------------------------------------------------------------------------------------------
# one pass
# ------------------------------------------------------------------------------------------
def _must(ok, what):
    if not ok:
        raise RuntimeError("step failed: %s" % (what,))


def _flow(c):
    """Velocity, pressure and positions after the pass."""
    q, k = c.get_state(), c.dim * c.N
    return dict(v=q[:k], p=q[k:k + c.N], x=c.get_positions())


def run(state):
    case, f = state["case"], state["case"]["family"]
    if f == "serving":
        return _serve(state)
    c = state["c"]
    if f == "newmesh":
        c.set_mesh_from(state["mesher"])
        _must(c.solve(case["dt"]), c.last_stats)
        return _flow(c)
    c.set_state(state["q"])
    if f == "heat":
        for _ in range(case["steps"]):
            _must(c.solve(state["dt"]), c.last_stats)
        return c.get_state()
    c.set_positions(state["pos"])
    if f == "wc":
        for _ in range(case["steps"]):
            c.solveOneTimeStep(c.computeNextDT(WC_SC, WC_MAXDT))
        return _wc_out(c)
    for _ in range(case["steps"]):
        _must(c.solve(case["dt"] if f == "pspg" else state["dt"]), c.last_stats)
    return _flow(c)


def _wc_out(c):
    q, k = c.get_state(), c.dim * c.N
    return dict(v=q[:k], p=q[k:k + c.N], rho=q[k + c.N:k + 2 * c.N], a=q[k + 2 * c.N:], x=c.get_positions())


def _serve(state):
    reqs, srv = state["reqs"], state["srv"]
    for r in reqs:
        r["c"].set_state(r["q"])
        r["c"].set_positions(r["mesh"].pos)
    for i, r in enumerate(reqs):
        srv.submit(r["c"], r["dt"], tag=i)
    left = len(reqs)
    while left:
        for res in srv.poll(timeout_ms=100):
            _must(res["status"] == 0, res)
            left -= 1
    out = {}
    for r in reqs:
        pre = "wc_" if r["kind"] == "WC" else ""
        for k, v in (_wc_out(r["c"]) if r["kind"] == "WC" else _flow(r["c"])).items():
            if pre and k == "a":
                continue  # the acceleration is the velocity's change, which is returned
            out.setdefault(pre + k, []).append(v.reshape(-1))
    return {k: np.concatenate(v) for k, v in out.items()}


# ------------------------------------------------------------------------------------------
# what a pass cannot do without, and how far two right answers lie apart
# ------------------------------------------------------------------------------------------
def _size(case):
    """(nodes, elements) of a case, as the mesh generators make them."""
    f, dim = case["family"], case.get("dim")
    if f in ("heat", "frac"):
        n = case["n"]
        return (n + 1) ** dim, n ** dim * (2 if dim == 2 else 6)
    N = case["nodes"]
    return N, 2 * N if dim == 2 else 6 * N


def work(case):
    """Mesh and node states read and written once per step; per element the products of its local
    matrices (incompressible, heat) or of its nodal sums (compressible)."""
    if case["family"] == "serving":
        b = fl = 0
        rng = np.random.default_rng([case["requests"], case["lo"], case["hi"]])
        for i in range(case["requests"]):
            dim = 2 if rng.random() < 0.6 else 3
            size = int(math.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"]))))
            w = work(dict(family="pspg" if i % 2 == 0 else "wc", dim=dim, nodes=size, state="fp32", steps=1))
            b, fl = b + w["bytes"], fl + w["flops"]
        return {"bytes": b, "flops": fl}
    N, E = _size(case)
    dim, steps = case["dim"], case.get("steps", 1)
    per_node = dict(pspg=dim + 1, newmesh=dim + 1, frac=dim + 1, heat=1, wc=2 * dim + 2)[case["family"]]
    s = 4 if case.get("state") == "fp32" else 8
    one = E * (dim + 1) * 4 + N * (1 + 2 * per_node * s + 2 * dim * 8)
    ne = dim + 1
    flops = E * (ne * ne * ne * ne * 2 if case["family"] in ("pspg", "newmesh", "frac") else ne * ne * 2 * dim + 60)
    return {"bytes": steps * one, "flops": steps * flops}


def tolerance(case):
    """About four times the largest difference seen between runs of the same inputs with other
    preconditioner settings and sums in another order, and from ``exact``: linear solves stop at
    relres 1e-10 (the stream: 1e-8), FP32 states round once per step."""
    f = case["family"]
    if f == "wc":
        return {"rel": 6e-6, "max": 1e-4} if case["state"] == "fp32" else {"rel": 1e-12, "max": 2e-11}
    if f == "serving":
        return {"rel": 2e-6, "max": 2e-5}
    if f in ("heat", "frac"):
        return {"rel": 4e-9, "max": 1e-7}
    return {"rel": 8e-7, "max": 5e-6}


# ------------------------------------------------------------------------------------------
# the same passes in plain torch, FP64
# ------------------------------------------------------------------------------------------
class _P1:
    """P1 elements of one mesh: connectivity, and geometry at given positions."""

    def __init__(self, conn, N, dim):
        self.dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
        self.conn = torch.as_tensor(np.ascontiguousarray(conn), dtype=torch.int64, device=self.dev)
        self.N, self.D, self.NE = N, dim, dim + 1

    def t(self, a):
        return torch.as_tensor(np.ascontiguousarray(a), device=self.dev)

    def geometry(self, pos):
        """(gN [E, a, k], |e|, det J, x [E, a, k])."""
        x = pos.t()[self.conn]
        J = (x[:, 1:] - x[:, :1]).transpose(1, 2)  # J[k][c]
        if self.D == 2:
            dj = J[:, 0, 0] * J[:, 1, 1] - J[:, 0, 1] * J[:, 1, 0]
            adj = torch.stack([torch.stack([J[:, 1, 1], -J[:, 0, 1]], 1), torch.stack([-J[:, 1, 0], J[:, 0, 0]], 1)], 1)
        else:
            c = [J[:, :, 0], J[:, :, 1], J[:, :, 2]]
            adj = torch.stack([torch.linalg.cross(c[1], c[2]), torch.linalg.cross(c[2], c[0]),
                               torch.linalg.cross(c[0], c[1])], 1)
            dj = (c[0] * adj[:, 0]).sum(1)
        g = adj / dj[:, None, None]
        return torch.cat([-g.sum(1, keepdim=True), g], 1), dj * (0.5 if self.D == 2 else 1 / 6), dj, x

    def scatter(self, v):
        """Sum of element-node values v [E, a, ...] over the nodes."""
        out = torch.zeros((self.N,) + v.shape[2:], dtype=v.dtype, device=self.dev)
        return out.index_add_(0, self.conn.reshape(-1), v.reshape((-1,) + v.shape[2:]))

    def graph(self):
        if not hasattr(self, "rows"):
            i = self.conn[:, :, None].expand(-1, -1, self.NE).reshape(-1)
            j = self.conn[:, None, :].expand(-1, self.NE, -1).reshape(-1)
            used = torch.zeros(self.N, dtype=torch.bool, device=self.dev)
            used[self.conn.reshape(-1)] = True
            self.free = ~used
            lone = torch.nonzero(self.free).reshape(-1)
            keys = torch.cat([i * self.N + j, lone * self.N + lone])
            u, inv = torch.unique(keys, return_inverse=True)
            self.rows, self.cols = u // self.N, u % self.N
            self.slot = inv[:i.numel()]
            self.diag = torch.searchsorted(u, torch.arange(self.N, device=self.dev) * (self.N + 1))
        return self

    def assemble(self, Ae):
        """Node-block values [entries, s, t] from element blocks Ae [E, a, b, s, t]."""
        self.graph()
        v = torch.zeros((self.rows.numel(),) + Ae.shape[3:], dtype=Ae.dtype, device=self.dev)
        return v.index_add_(0, self.slot, Ae.reshape((-1,) + Ae.shape[3:]))

    def mul(self, vals, x):
        """A x for node blocks vals [entries, s, t], x [N, t]."""
        y = torch.zeros((self.N, vals.shape[1]), dtype=x.dtype, device=self.dev)
        return y.index_add_(0, self.rows, (vals * x[self.cols][:, None, :]).sum(2))


def _bicgstab(P, A, b, x, rtol, most=20000):
    """Right-preconditioned (block Jacobi) BiCGSTAB, restarted on its true residual."""
    M = torch.linalg.inv(A[P.diag])
    pre = lambda r: (M * r[:, None, :]).sum(2)  # noqa: E731
    bb = float((b * b).sum())
    it, best, good = 0, math.inf, x
    for _ in range(40):
        r = b - P.mul(A, x)
        rr = float((r * r).sum())
        if rr < best:
            best, good = rr, x
        else:  # broken down: again from the best iterate
            x = good
            r = b - P.mul(A, x)
        if best <= rtol * rtol * bb or it >= most:
            break
        rh, rho = r.clone(), (r * r).sum()
        p = r.clone()
        while it < most:
            it += 1
            ph = pre(p)
            v = P.mul(A, ph)
            alpha = rho / (rh * v).sum()
            s = r - alpha * v
            sh = pre(s)
            t = P.mul(A, sh)
            om = (t * s).sum() / (t * t).sum()
            x = x + alpha * ph + om * sh
            r = s - om * t
            if it % 10 == 0:
                rr = float((r * r).sum())
                if not math.isfinite(rr) or rr <= 0.25 * rtol * rtol * bb:
                    break
            new = (rh * r).sum()
            p = r + (new / rho) * (alpha / om) * (p - om * v)
            rho = new
    return good


def _cg(P, A, b, x, rtol, most=20000):
    """Diagonal-preconditioned conjugate gradient."""
    d = torch.diagonal(A[P.diag], dim1=1, dim2=2)
    d = torch.where(d != 0, 1 / d, torch.ones_like(d))
    r = b - P.mul(A, x)
    z = d * r
    p, rz, bb = z.clone(), (r * z).sum(), float((b * b).sum())
    for it in range(most):
        if it % 5 == 0 and float((r * r).sum()) <= rtol * rtol * bb:
            break
        q = P.mul(A, p)
        alpha = rz / (p * q).sum()
        x = x + alpha * p
        r = r - alpha * q
        z = d * r
        new = (r * z).sum()
        p = z + (new / rz) * p
        rz = new
    return x


def _pspg_system(P, fl, pos, v_prev, v_it, dt, rho=1000.0, mu=1e-3):
    """Node blocks and right-hand side [N, d + 1] with the boundary conditions (walls at rest)."""
    D, NE, g = P.D, P.NE, torch.zeros(P.D, dtype=torch.float64, device=P.dev)
    g[D - 1] = -9.81
    gN, vol, dj, _ = P.geometry(pos)
    P.graph()
    h = torch.sqrt((0.5 if D == 2 else 1 / 6) * dj / math.pi)
    U = torch.sqrt((v_it[P.conn] ** 2).sum(2)).sum(1) / NE
    visc = 4 * mu / (h * h * rho)
    tau = 1 / torch.sqrt((2 / dt) ** 2 + (2 * U / h) ** 2 + 9 * visc ** 2)
    e = lambda w: w[:, None, None]  # noqa: E731
    gg = torch.einsum("eak,ebk->eab", gN, gN)
    mass = e(rho * vol / ((D + 1) * (D + 2))) * (1 + torch.eye(NE, dtype=torch.float64, device=P.dev))
    Ae = torch.zeros((P.conn.shape[0], NE, NE, NE, NE), dtype=torch.float64, device=P.dev)
    for s in range(D):
        for t in range(D):
            Ae[:, :, :, s, t] = e(mu * vol) * gN[:, :, None, t] * gN[:, None, :, s]
        Ae[:, :, :, s, s] += mass / dt + e(mu * vol) * gg
        Ae[:, :, :, s, D] = -e(vol / NE) * gN[:, :, None, s]
        Ae[:, :, :, D, s] = e(vol / NE) * (e(tau / dt) * gN[:, :, None, s] + gN[:, None, :, s])
    Ae[:, :, :, D, D] = e(tau / rho * vol) * gg
    vp = v_prev[P.conn]
    be = torch.zeros((P.conn.shape[0], NE, NE), dtype=torch.float64, device=P.dev)
    be[:, :, :D] = e(rho * vol / NE) * g + torch.einsum("eab,ebk->eak", mass / dt, vp)
    be[:, :, D] = (tau * vol)[:, None] * (gN @ g) + torch.einsum("eak,ek->ea", gN, vp.sum(1)) * (tau / dt * vol / NE)[:, None]
    A, b = P.assemble(Ae), P.scatter(be)
    del Ae, be
    bound = (fl & mg.BOUND) != 0
    for s in range(D):
        A[:, :, s] *= (~(bound & ~P.free))[P.cols].to(A.dtype)[:, None]   # eliminated wall columns (values 0)
        A[:, s, :] *= (~(bound | P.free))[P.rows].to(A.dtype)[:, None]    # unit rows
        A[P.diag, s, s] = torch.where(bound | P.free, torch.ones_like(b[:, s]), A[P.diag, s, s])
        b[:, s] = torch.where(bound, torch.zeros_like(b[:, s]), torch.where(P.free, v_prev[:, s] + dt * g[s], b[:, s]))
    A[P.diag, D, D] = torch.where(P.free, torch.ones_like(b[:, D]), A[P.diag, D, D])
    return A, b


def _pspg_exact(dim, conn, flags, pos, q, dt, steps):
    P = _P1(conn, pos.shape[1], dim)
    fl = P.t(flags)
    x, q = P.t(pos), P.t(q).reshape(dim + 1, -1).t().contiguous()
    fixed = (fl & mg.FIXED) != 0
    for _ in range(steps):
        x0, prev, it = x.clone(), q.clone(), 0
        A, b = _pspg_system(P, fl, x, prev[:, :dim], q[:, :dim], dt)
        res = math.inf
        while res > 1e-6 and it <= 10:
            q = _bicgstab(P, A, b, q, 1e-12)
            x = torch.where(fixed, x0, x0 + dt * q[:, :dim].t())
            A, b = _pspg_system(P, fl, x, prev[:, :dim], q[:, :dim], dt)
            res = float((P.mul(A, q) - b).norm())
            it += 1
    q = q.t().contiguous().cpu().numpy()
    return dict(v=q[:dim].reshape(-1), p=q[dim], x=x.cpu().numpy())


def _wc_exact(dim, conn, flags, pos, q, steps):
    P = _P1(conn, pos.shape[1], dim)
    N, D, NE, mu = P.N, dim, dim + 1, 1e-3
    fl, x, q = P.t(flags), P.t(pos), P.t(q)
    v, p, rho, a = (q[:D * N].reshape(D, N), q[D * N:(D + 1) * N], q[(D + 1) * N:(D + 2) * N],
                    q[(D + 2) * N:].reshape(D, N))
    fixed, bound = (fl & mg.FIXED) != 0, (fl & mg.BOUND) != 0
    g = torch.zeros(D, dtype=torch.float64, device=P.dev)
    g[D - 1] = -9.81
    c2 = 1.0 / ((D + 1) * (D + 2))

    def h_e(xe, vol):
        n = lambda i, j: (xe[:, i] - xe[:, j]).norm(dim=1)  # noqa: E731
        if D == 2:
            return 2 * vol / ((n(0, 1) + n(1, 2) + n(0, 2)) / 2)
        f = lambda i, j, k: torch.linalg.cross(xe[:, j] - xe[:, i], xe[:, k] - xe[:, i]).norm(dim=1)  # noqa: E731
        return 12 * vol / (f(0, 1, 2) + f(0, 3, 2) + f(0, 1, 3) + f(3, 1, 2))

    def next_dt(he):
        u2, al = (v * v).sum(0)[P.conn], (mu / rho)[P.conn]
        S = torch.maximum(torch.maximum(u2, ((K0 + K0P * p) / rho)[P.conn]), 4 * al * al / (he * he)[:, None]).amax(1)
        return min(math.sqrt(float((WC_SC ** 2 * he * he / S).min())), WC_MAXDT)

    gN, vol, _, xe = P.geometry(x)
    dt = next_dt(h_e(xe, vol))
    for _ in range(steps):
        v = v + 0.5 * dt * a
        x = torch.where(fixed, x, x + dt * v)
        gN, vol, _, xe = P.geometry(x)
        ve, pe = v.t()[P.conn], p[P.conn]
        div = (gN * ve).sum((1, 2))
        ps = pe + pe.sum(1, keepdim=True)
        w = vol[:, None]
        f = -dt * w * (K0 / NE + K0P * ps * c2) * div[:, None] + w * ps * c2
        p = P.scatter(f) / P.scatter((w / NE).expand(-1, NE))
        rho = ((K0P / K0) * p + 1.0) ** (1.0 / K0P) * RHO0
        re, psum = rho[P.conn], p[P.conn].sum(1)
        L = torch.einsum("eam,eak->ekm", gN, ve)
        sig = L + L.transpose(1, 2) - (2.0 / 3.0) * torch.diagonal(L, dim1=1, dim2=2).sum(1)[:, None, None] * \
            torch.eye(D, dtype=torch.float64, device=P.dev)
        ml = w * (re + re.sum(1, keepdim=True)) * c2
        F = -(mu * vol)[:, None, None] * torch.einsum("eam,esm->eas", gN, sig) + (vol * psum / NE)[:, None, None] * gN \
            + ml[:, :, None] * g
        a = (P.scatter(F) / P.scatter(ml)[:, None]).t()
        a = torch.where(bound, torch.zeros_like(a), a)
        v = v + 0.5 * dt * a
        dt = next_dt(h_e(xe, vol))
    c = lambda z: z.reshape(-1).cpu().numpy()  # noqa: E731
    return dict(v=c(v), p=c(p), rho=c(rho), a=c(a), x=x.cpu().numpy())


def _heat_exact(dim, m, T0, Tbc, dt, steps):
    P = _P1(m.conn, m.n_nodes, dim)
    dirichlet = (P.t(m.flags) & mg.DIRICHLET) != 0
    T, Tb = P.t(T0)[:, None], P.t(Tbc)[:, None]
    gN, vol, _, _ = P.geometry(P.t(m.pos))
    mass = (HEAT_MAT["rho"] * HEAT_MAT["cv"] * vol / ((dim + 1) * (dim + 2)))[:, None, None] * \
        (1 + torch.eye(P.NE, dtype=torch.float64, device=P.dev))
    lap = (HEAT_MAT["k"] * vol)[:, None, None] * torch.einsum("eak,ebk->eab", gN, gN)
    A0, M0 = P.assemble((mass + dt * lap)[..., None, None]), P.assemble(mass[..., None, None])
    A = A0 * (~dirichlet[P.rows] & ~dirichlet[P.cols]).to(A0.dtype)[:, None, None]
    A[P.diag, 0, 0] = torch.where(dirichlet, torch.ones_like(T[:, 0]), A0[P.diag, 0, 0])
    lift = P.mul(A0, torch.where(dirichlet[:, None], Tb, torch.zeros_like(Tb)))
    for _ in range(steps):
        T = _cg(P, A, torch.where(dirichlet[:, None], Tb, P.mul(M0, T) - lift), T, 1e-14)
    return T[:, 0].cpu().numpy()


def _frac_exact(dim, m, q, vbc, dt, steps):
    P = _P1(m.conn, m.n_nodes, dim)
    kw = _frac_kw(dim)
    rho, mu, D = kw["rho"], kw["mu"], dim
    bound = ((P.t(m.flags) & mg.BOUND) != 0)[:, None]
    vb, q = P.t(vbc).t().contiguous(), P.t(q).reshape(dim + 1, -1).t()
    g = torch.tensor(kw["body_force"], dtype=torch.float64, device=P.dev)
    x, v, p = P.t(m.pos), q[:, :D].contiguous(), q[:, D:].contiguous()
    inner = (~bound[:, 0])
    eye = torch.eye(D, dtype=torch.float64, device=P.dev)
    for _ in range(steps):
        x0, v0, p0, vi, it, res = x.clone(), v.clone(), p.clone(), v.clone(), 0, math.inf
        while res > 1e-6 and it <= 10:
            gN, vol, _, _ = P.geometry(x)
            w = vol[:, None, None]
            gg = torch.einsum("eak,ebk->eab", gN, gN)
            mass = rho * w / ((D + 1) * (D + 2)) * (1 + torch.eye(P.NE, dtype=torch.float64, device=P.dev))
            K = (mu * w)[..., None, None] * (gg[..., None, None] * eye + torch.einsum("eac,ebr->eabrc", gN, gN))
            MK = P.assemble(mass[..., None, None] / dt * eye + K)
            del K
            ms, L = P.assemble(mass[..., None, None]), P.assemble(w[..., None, None] * gg[..., None, None])
            lift = P.mul(MK, torch.where(bound, vb, torch.zeros_like(vb)))
            be = rho * g * (vol / P.NE)[:, None, None] + torch.einsum("eab,ebk->eak", mass / dt, v0[P.conn]) + \
                w / P.NE * gN * p0[P.conn].sum(1, keepdim=True)
            b = torch.where(bound, vb, P.scatter(be) - lift)
            keep = (inner[P.rows] & inner[P.cols]).to(MK.dtype)[:, None, None]
            unit = torch.where(bound[:, :, None], eye, torch.zeros_like(MK[P.diag]))
            MK, ms = MK * keep, ms * keep
            MK[P.diag] += unit
            ms[P.diag] += unit[:, :1, :1]
            vt = _cg(P, MK, b, torch.zeros_like(b), 1e-14)
            bp = P.scatter(-(rho / dt) * w[:, :, 0] / P.NE * torch.einsum("eak,eak->e", gN, vt[P.conn])[:, None].expand(-1, P.NE))
            pn = _cg(P, L, (bp + P.mul(L, p0)[:, 0])[:, None], torch.zeros_like(p0), 1e-13)
            bv = dt * P.scatter(w / P.NE * gN * (pn - p0)[P.conn].sum(1, keepdim=True))
            bv = torch.where(bound, torch.zeros_like(bv), bv)
            dv = torch.cat([_cg(P, ms, bv[:, k:k + 1].contiguous(), torch.zeros_like(p0), 1e-14) for k in range(D)], 1)
            v = vt + dv
            x = torch.where(bound[:, 0], x0, x0 + dt * v.t())
            prev2 = float((vi * vi).sum())
            res = math.sqrt(float(((v - vi) ** 2).sum()) / prev2) if prev2 else math.inf
            vi, p, it = v.clone(), pn, it + 1
    c = lambda z: z.t().reshape(-1).cpu().numpy()  # noqa: E731
    return dict(v=c(v), p=c(p), x=x.cpu().numpy())


def exact(case, seed):
    f, dim = case["family"], case.get("dim")
    if f == "pspg":
        m = _mesh(case["mesh"], dim, case["nodes"], seed)
        return _pspg_exact(dim, m.conn, m.flags, m.pos, _pspg_state(m, seed), case["dt"], case["steps"])
    if f == "newmesh":
        t = _newmesh_cloud(case, seed)
        pos, q, fl, _ = t.nodes()
        return _pspg_exact(dim, t.elements(), fl, pos, q.reshape(-1), case["dt"], 1)
    if f == "wc":
        if _size(case)[1] * case["steps"] > 1.3e9:
            return None
        m = _mesh("tank", dim, case["nodes"], seed)
        return _wc_exact(dim, m.conn, m.flags, m.pos, _wc_state(m, seed), case["steps"])
    if f == "heat":
        m, T0, Tbc, dt = _heat_inputs(case, seed)
        return _heat_exact(dim, m, T0, Tbc, dt, case["steps"])
    if f == "frac":
        m, q, vbc, dt = _frac_inputs(case, seed)
        return _frac_exact(dim, m, q, vbc, dt, case["steps"])
    return None  # the stream's many solves take longer than a reference run should
