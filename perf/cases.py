"""The cases that the framework's speed is measured on.

Every case is one of the package's device entry points as a program that uses
it calls them: `Plan.matvec_torch` (the reference's feMatrix::matVec /
fem::matvec), `Plan.cg_solve_torch`, `Plan.bicgstab_solve_torch`,
`cg_solve_batch_torch` (the serving layer's batched solves) and `Batch` (many
meshes in one graph replay).  Meshes are the two families of the
benchmark and the tests: 2:1 balanced trees refined around a sphere (dim 2 and
3) and trees of Gaussian-mixture points (dim 4, and 2 or 3 in draws), from
about a thousand elements to the 15.3M elements of the headline workload.

Solves run a fixed number of iterations from x = 0 (tolerance 0), so a pass is
the same work whatever the rounding, and few enough that the iteration has not
yet amplified it (a perturbation of 2e-16 in every product grows to at most
5e-13 in x within 24 CG iterations on these meshes, and to 1e-2 within 64;
BiCGStab: 1e-13 within 8); FP64 throughout, as the solution of an
FP32 iteration is only defined to its own accuracy before it has converged
(FP32 is covered by the matvecs it is made of).

A mesh is fixed by its case; the vectors come from the seed.  The host mesh is
kept between preparations (a program makes it once); every state has a device
plan of its own.
"""
import functools
import importlib.util
import math
import os
import random
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _module(name, file):
    if name not in sys.modules:
        spec = importlib.util.spec_from_file_location(name, os.path.join(ROOT, "dendro-kt_amd", file))
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name]


dkt = _module("dkt", "__init__.py")
spacetime = _module("dkt_spacetime", "spacetime.py")

MAXD = {2: 30, 3: 30, 4: 9}  # tree depth limit per dimension, as in the benchmark's workloads


# ---------------------------------------------------------------------------
# Cases.
# ---------------------------------------------------------------------------
def listed():
    centre = dict(cx=0.5, cy=0.5, cz=0.5, radius=0.3)
    return [
        # The headline: Poisson on a 4D space-time tree of 2e6 points, the
        # reference's traversal semantics, FP64 and FP32.
        dict(name="matvec-4d-2m-f64", kind="matvec", dim=4, p=1, points=2000000, mesh_seed=1, conforming=False,
             op="stiffness", dtype="f64", masked=0, nrhs=1),
        dict(name="matvec-4d-2m-f32", kind="matvec", dim=4, p=1, points=2000000, mesh_seed=1, conforming=False,
             op="stiffness", dtype="f32", masked=0, nrhs=1),
        # The smallest call: a 3D tree of about a thousand elements with
        # Dirichlet hooks, where launches and latency are all there is.
        dict(name="matvec-3d-1k-f64", kind="matvec", dim=3, p=1, base=2, level=5, conforming=False, op="stiffness",
             dtype="f64", masked=1, nrhs=1, cx=0.43, cy=0.52, cz=0.47, radius=0.17),
        # The reference's own kind of run: 3D, p = 1, level 7 (82,776 elements).
        dict(name="matvec-3d-l7-f64", kind="matvec", dim=3, p=1, base=3, level=7, conforming=False, op="stiffness",
             dtype="f64", masked=0, nrhs=1, **centre),
        # Quadratic elements, eight right-hand sides interleaved per node, FP32.
        dict(name="matvec-3d-p2-8rhs-f32", kind="matvec", dim=3, p=2, base=3, level=7, conforming=False,
             op="stiffness", dtype="f32", masked=0, nrhs=8, **centre),
        # The operator of the level-9 p = 2 solve (8.9M nodes), conforming, masked.
        dict(name="matvec-3d-p2-l9-conf-f64", kind="matvec", dim=3, p=2, base=3, level=9, conforming=True,
             op="stiffness", dtype="f64", masked=1, nrhs=1, **centre),
        # Many independent trees (p = 1 and 2 in turn, 8 right-hand sides each,
        # one column after another), one graph replay.
        dict(name="batch-32-8rhs-f32", kind="batch", trees=32, lo=1000, hi=200000, mesh_seed=3, nrhs=8, dtype="f32"),
        # Served solves: a small conforming 3D mesh alone (latency per iteration),
        dict(name="cg-3d-conf-6k", kind="cg", dim=3, p=1, base=2, level=6, conforming=True, iters=24,
             cx=0.43, cy=0.52, cz=0.47, radius=0.17),
        # the benchmark's 4D solve on the reference's operator (176k nodes),
        dict(name="cg-4d-20k", kind="cg", dim=4, p=1, points=20000, mesh_seed=2, conforming=False, iters=64),
        # the large p = 2 solve (8.9M nodes),
        dict(name="cg-3d-p2-l9", kind="cg", dim=3, p=2, base=3, level=9, conforming=True, iters=32, **centre),
        # eight meshes of the serving pool's sizes solved together,
        dict(name="cg-batch-8", kind="cgbatch", meshes=8, lo=1000, hi=200000, mesh_seed=0, iters=24),
        # and the stabilised space-time heat form (captured element matrices).
        dict(name="bicgstab-4d-2k", kind="bicgstab", points=2000, mesh_seed=5, iters=8),
    ]


def draw(rng):
    def log_uniform(lo, hi):
        return math.exp(rng.uniform(math.log(lo), math.log(hi)))

    def mesh(dim, target):
        if dim == 4 or rng.random() < 0.25:  # points: about 15 elements per point in 4D, 4 in 2D and 3D
            return dict(points=max(40, int(target / (10 if dim == 4 else 4))), mesh_seed=rng.randrange(1000))
        radius = round(rng.uniform(0.1, 0.3), 3)
        per = 58.0 * radius * radius if dim == 3 else 30.0 * radius  # elements of the refined band per 4^level (2^level)
        level = max(4, min(14 if dim == 2 else 9, int(round(math.log(target / per, 4 if dim == 3 else 2)))))
        out = dict(base=rng.choice([2, 3]), level=level, radius=radius, cx=round(rng.uniform(0.3, 0.7), 3),
                   cy=round(rng.uniform(0.3, 0.7), 3))
        return dict(out, cz=round(rng.uniform(0.3, 0.7), 3)) if dim == 3 else out

    what = rng.random()
    if what < 0.55:
        dim = rng.choice([2, 3, 3, 4, 4])
        p = 1 if dim == 4 else rng.choice([1, 1, 2])
        m = mesh(dim, log_uniform(1e3, 1e6 / (1 if p == 1 else 4)))
        return dict(kind="matvec", dim=dim, p=p, conforming=rng.random() < 0.4,
                    op=rng.choice(["stiffness", "stiffness", "mass"]), dtype=rng.choice(["f64", "f64", "f32"]),
                    masked=rng.choice([0, 1, 1, 2]), nrhs=rng.choice([1, 1, 1, 2, 3, 8]), **m)
    if what < 0.8:
        dim = rng.choice([3, 3, 4])
        p = 1 if dim == 4 else rng.choice([1, 1, 2])
        m = mesh(dim, log_uniform(1e3, 3e5 / (1 if p == 1 else 4)))
        return dict(kind="cg", dim=dim, p=p, conforming=dim == 3 or rng.random() < 0.5, iters=rng.choice([8, 16, 24]), **m)
    if what < 0.9:
        return dict(kind="batch", trees=rng.randint(5, 24), lo=1000, hi=int(log_uniform(1e4, 1e5)),
                    mesh_seed=rng.randrange(1000), nrhs=rng.choice([1, 3, 8]), dtype=rng.choice(["f32", "f64"]))
    if what < 0.96:
        return dict(kind="cgbatch", meshes=rng.randint(2, 7), lo=1000, hi=int(log_uniform(1e4, 1e5)),
                    mesh_seed=rng.randrange(1000), iters=rng.choice([8, 16, 24]))
    return dict(kind="bicgstab", points=int(log_uniform(100, 4000)), mesh_seed=rng.randrange(1000), iters=8)


# ---------------------------------------------------------------------------
# Meshes.
# ---------------------------------------------------------------------------
def _da(case, p=None):
    keys = ("dim", "points", "mesh_seed", "base", "level", "cx", "cy", "cz", "radius")
    return _mesh(case.get("p", 1) if p is None else p, tuple((k, case[k]) for k in keys if k in case))


@functools.lru_cache(maxsize=6)
def _mesh(p, items):
    m = dict(items)
    dim = m["dim"]
    if "points" in m:
        cells = dkt.gauss_points(dim, 9, m["points"], 4, 0.05, m["mesh_seed"])
    else:
        cells = dkt.sphere_tree(dim, MAXD[dim], m["base"], m["level"], [m[k] for k in ("cx", "cy", "cz")[:dim]],
                                m["radius"])
    da = dkt.DA(dkt.balance_tree(cells, 1), p)
    da.maxd = 9 if "points" in m else MAXD[dim]
    return da


@functools.lru_cache(maxsize=2)
def _pool(kind, n, lo, hi, seed):
    """[(mesh, order)]: n trees, element counts about log-uniform in [lo, hi].
    batch: 3D spheres, p alternating 1 and 2; serve: p = 1, 70% 3D spheres,
    30% 4D Gaussian mixtures."""
    rng = random.Random(seed)
    out = []
    for k in range(n):
        target = lo * (hi / lo) ** ((k + rng.random()) / n)
        four = kind == "serve" and rng.random() >= 0.7
        radius, c = rng.uniform(0.1, 0.3), [rng.uniform(0.2, 0.8) for _ in range(3)]
        p = 1 + k % 2 if kind == "batch" else 1
        if four:
            m = dict(dim=4, points=max(50, int(2000 * (target / 31261.0) ** (1 / 0.89))), mesh_seed=1000 + k)
        else:
            level = max(3, int(round(math.log(target / (58.0 * radius * radius), 4))))
            m = dict(dim=3, base=2, level=level, cx=c[0], cy=c[1], cz=c[2], radius=radius)
        out.append(_mesh.__wrapped__(p, tuple(m.items())))
    return out


OPS = {"stiffness": dkt.OP_STIFFNESS, "mass": dkt.OP_MASS}
DTYPE = {"f64": torch.float64, "f32": torch.float32}


def _rand(shape, gen, dtype=torch.float64):
    """uniform[-1, 1], the input of every configuration."""
    return torch.rand(shape, generator=gen, device="cuda", dtype=dtype) * 2 - 1


def _rhs(da, gen):
    """A right-hand side with Dirichlet zero boundary."""
    b = _rand(da.n_nodes, gen)
    b[torch.from_numpy(da.boundary().astype(np.int64)).cuda()] = 0.0
    return b


def _captured(da):
    ids = spacetime.dirichlet_nodes(da.nodes(), da.maxd)
    return spacetime.level_matrices(da.maxd), ids


@functools.lru_cache(maxsize=1)
def _stream():
    """A graph replays on a stream of its own, which the program keeps."""
    return torch.cuda.Stream()


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    kind = case["kind"]
    if kind == "matvec":
        da = _da(case)
        shape = (da.n_nodes,) if case["nrhs"] == 1 else (da.n_nodes, case["nrhs"])
        x = _rand(shape, gen, DTYPE[case["dtype"]])
        plan = dkt.Plan(da, OPS[case["op"]], conforming=case["conforming"])
        return dict(case=case, plan=plan, x=x, y=torch.empty_like(x))
    if kind == "cg":
        da = _da(case)
        b = _rhs(da, gen)
        return dict(case=case, plan=dkt.Plan(da, conforming=case["conforming"]), b=b, x=torch.empty_like(b))
    if kind == "bicgstab":
        da = _da(dict(case, dim=4))
        mats, ids = _captured(da)
        plan = dkt.Plan(da, dkt.OP_CAPTURED, mats, conforming=True)
        plan.set_dirichlet(ids)
        b = _rand(da.n_nodes, gen)
        b[torch.from_numpy(ids.astype(np.int64)).cuda()] = 0.0
        return dict(case=case, plan=plan, b=b, x=torch.empty_like(b))
    if kind == "cgbatch":
        das = _pool("serve", case["meshes"], case["lo"], case["hi"], case["mesh_seed"])
        bs = [_rhs(da, gen) for da in das]
        return dict(case=case, plans=[dkt.Plan(da, conforming=True) for da in das], b=bs,
                    x=[torch.empty_like(b) for b in bs])
    das = _pool("batch", case["trees"], case["lo"], case["hi"], case["mesh_seed"])
    xs = [_rand((case["nrhs"], da.n_nodes), gen, DTYPE[case["dtype"]]) for da in das]
    ys = [torch.empty_like(x) for x in xs]
    plans = [dkt.Plan(da) for da in das]
    return dict(case=case, batch=dkt.Batch(plans, xs, ys, graph=True, column_major=True), y=ys, stream=_stream())


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "matvec":
        state["plan"].matvec_torch(state["x"], state["y"], masked=case["masked"])
        return state["y"]
    if kind == "batch":
        state["batch"].run(state["stream"].cuda_stream)
        return state["y"]
    if kind == "cgbatch":
        dkt.cg_solve_batch_torch(state["plans"], state["b"], state["x"], max_iter=case["iters"], tol=0.0)
        return state["x"]
    state["x"].zero_()
    if kind == "cg":
        state["plan"].cg_solve_torch(state["b"], state["x"], dkt.CG_F64, case["iters"], 0.0)
    else:
        state["plan"].bicgstab_solve_torch(state["b"], state["x"], case["iters"], 0.0)
    return state["x"]


# ---------------------------------------------------------------------------
# Work: x read and y written once, and per element one 16-bit index for each
# of its nodes and its level; the element product by axes (2 nPe (p + 1) per
# axis there and back).  An iteration of a solve adds its vectors: CG reads
# and writes x, r and p and reads A p.
# ---------------------------------------------------------------------------
def _matvec_work(da, size, nrhs):
    npe, E = da.npe, da.n_elements
    return 2.0 * size * nrhs * da.n_nodes + E * (2.0 * npe + 1), nrhs * E * 4.0 * da.dim * npe * (da.order + 1)


def work(case):
    kind, size = case["kind"], 4 if case.get("dtype") == "f32" else 8
    if kind == "matvec":
        by, fl = _matvec_work(_da(case), size, case["nrhs"])
    elif kind == "batch":
        das = _pool("batch", case["trees"], case["lo"], case["hi"], case["mesh_seed"])
        by, fl = (sum(v) for v in zip(*(_matvec_work(da, size, case["nrhs"]) for da in das)))
    else:
        das = _pool("serve", case["meshes"], case["lo"], case["hi"], case["mesh_seed"]) if kind == "cgbatch" else \
            [_da(dict(case, dim=case.get("dim", 4)))]
        by = fl = 0.0
        for da in das:
            b, f = _matvec_work(da, 8, 1)
            mv, vec = (2, 12 * 8.0) if kind == "bicgstab" else (1, 5 * 8.0)  # vectors besides the matvec's own two
            by += case["iters"] * (mv * b + vec * da.n_nodes)
            fl += case["iters"] * (mv * f + (20.0 if kind == "bicgstab" else 10.0) * da.n_nodes)
    return {"bytes": by, "flops": fl}


# ---------------------------------------------------------------------------
# Exact values: the operators in plain torch, 64 bits.
# ---------------------------------------------------------------------------
def _one_d(p):
    if p == 1:
        return np.array([[1.0, -1.0], [-1.0, 1.0]]), np.array([[2.0, 1.0], [1.0, 2.0]]) / 6.0
    return (np.array([[7.0, -8.0, 1.0], [-8.0, 16.0, -8.0], [1.0, -8.0, 7.0]]) / 3.0,
            np.array([[4.0, 2.0, -1.0], [2.0, 16.0, 2.0], [-1.0, 2.0, 4.0]]) / 30.0)


def _kron(mats):
    """Tensor product, axis 0 fastest."""
    out = np.array([[1.0]])
    for m in mats:
        out = np.kron(m, out)
    return out


def _element(dim, p, op):
    """Element matrix of the unit cube and its power of the element size."""
    K, M = _one_d(p)
    if op == "mass":
        return _kron([M] * dim), dim
    return sum(_kron([K if d == t else M for d in range(dim)]) for t in range(dim)), dim - 2


def _interp(p, c):
    """W[i, k]: weight of parent node k at node i of child half c."""
    t = np.arange(p + 1) / p
    at = 0.5 * (c + t)
    w = np.ones((p + 1, p + 1))
    for k in range(p + 1):
        for j in range(p + 1):
            if j != k:
                w[:, k] *= (at - t[j]) / (t[k] - t[j])
    return w


def _dev(a, kind=None):
    return torch.from_numpy(np.ascontiguousarray(a if kind is None else a.astype(kind))).cuda()


class _Reference:
    """fem::matvec over the mesh's traversal (leaves, their nodes, the parent
    nodes of hanging leaves and the terms of the stale parent buffer)."""

    def __init__(self, da, op):
        tr = da.traversal()
        dim, p, self.npe = da.dim, da.order, da.npe
        K, hp = _element(dim, p, op)
        self.K = _dev(K.T)
        self.scale = _dev(2.0 ** (-hp * tr["cells"][:, dim].astype(np.float64)))
        self.slot = _dev(tr["slot"], np.int64)
        hang = _dev(tr["hang_of"], np.int64)
        self.hl = torch.nonzero(hang >= 0).flatten()  # hanging leaves, by hanging index
        self.ps = _dev(tr["pslot"], np.int64)
        child = _dev(tr["child"], np.int64)[self.hl]
        self.by_child = [(torch.nonzero(child == c).flatten(), _kron([_interp(p, (c >> d) & 1) for d in range(dim)]))
                         for c in range(1 << dim)]
        self.by_child = [(i, _dev(w.T), _dev(w)) for i, w in self.by_child if i.numel()]
        count = np.diff(tr["hc_off"])
        self.st = (_dev(np.repeat(np.arange(len(count)) * self.npe, count) + tr["hc_rank"]),
                   _dev(tr["hc_node"], np.int64), _dev(tr["hc_w"]))

    def __call__(self, x):
        def gather(s):
            return torch.where(s >= 0, x[s.clamp(min=0)], x.new_zeros(()))
        u = gather(self.slot)
        hs = self.slot[self.hl]
        par = gather(self.ps)
        ui = torch.empty_like(par)
        for i, wt, _ in self.by_child:
            ui[i] = par[i] @ wt
        ui.view(-1).index_add_(0, self.st[0], self.st[2] * x[self.st[1]])
        u[self.hl] = torch.where(hs >= 0, u[self.hl], ui)
        v = (u @ self.K) * self.scale[:, None]
        y = torch.zeros_like(x)
        on = self.slot >= 0
        y.index_add_(0, self.slot[on], v[on])
        vm = torch.where(hs >= 0, v.new_zeros(()), v[self.hl])
        for i, _, w in self.by_child:
            ui[i] = vm[i] @ w
        to = (self.ps >= 0) & (hs < 0)
        y.index_add_(0, self.ps[to], ui[to])
        return y


class _Conforming:
    """sum_e C_e^T K_e C_e: a rank of an element that is no node takes the
    parent cell's interpolant, and so on until every point is a node."""

    def __init__(self, da, op=None, mats=None):
        dim, p, maxd, self.npe = da.dim, da.order, da.maxd, da.npe
        nodes, cells = da.nodes().astype(np.int64), da.elements().astype(np.int64)
        lev, n1 = cells[:, dim], p + 1
        if mats is None:
            K, hp = _element(dim, p, op)
            self.levels = [(slice(None), _dev(K.T))]
            self.scale = _dev(2.0 ** (-hp * lev.astype(np.float64)))
        else:
            self.levels = [(_dev(np.nonzero(lev == k)[0]), _dev(mats[k].T)) for k in np.unique(lev)]
            self.scale = torch.ones(len(cells), dtype=torch.float64, device="cuda")
        big = (1 << maxd) + 1

        def key(x):  # coordinates as one number (a hash in wrapping arithmetic where they do not fit)
            k = np.zeros(x.shape[0], np.uint64)
            for d in range(dim):
                k = k * np.uint64(big if dim * maxd < 62 else 0x9E3779B97F4A7C15) + x[:, d].astype(np.uint64)
            return k
        nk = key(nodes[:, :dim])
        order = np.argsort(nk)
        nk = nk[order]
        digits = np.stack([(np.arange(self.npe) // n1 ** d) % n1 for d in range(dim)], 1)
        step = (1 << (maxd - lev)) // p
        E = len(cells)
        org = np.repeat(cells[:, :dim], self.npe, 0)
        pos = org + (step[:, None, None] * digits[None]).reshape(-1, dim)
        row, lv, wt = np.arange(E * self.npe), np.repeat(lev, self.npe), np.ones(E * self.npe)
        ip = [_interp(p, 0), _interp(p, 1)]
        rows, cols, vals = [], [], []
        while len(row):
            k = key(pos)
            at = np.minimum(np.searchsorted(nk, k), len(nk) - 1)
            hit = nk[at] == k
            rows.append(row[hit])
            cols.append(order[at[hit]])
            vals.append(wt[hit])
            row, lv, wt, pos, org = (a[~hit] for a in (row, lv, wt, pos, org))
            ln = 1 << (maxd - lv)
            par = org & ~(2 * ln - 1)[:, None]
            c = (org - par) // ln[:, None]
            t = (pos - org) // (ln // p)[:, None]
            nxt = []
            for u in range(self.npe):
                w = wt.copy()
                for d in range(dim):
                    w *= np.where(c[:, d] == 0, ip[0][t[:, d], digits[u, d]], ip[1][t[:, d], digits[u, d]])
                on = w != 0
                nxt.append((row[on], lv[on] - 1, w[on], par[on] + (2 * ln[on] // p)[:, None] * digits[u], par[on]))
            row, lv, wt, pos, org = (np.concatenate(a) for a in zip(*nxt))
        self.rows, self.cols = _dev(np.concatenate(rows)), _dev(np.concatenate(cols))
        self.vals = _dev(np.concatenate(vals))
        self.E = E

    def __call__(self, x):
        u = x.new_zeros(self.E * self.npe).index_add_(0, self.rows, self.vals * x[self.cols]).view(self.E, self.npe)
        v = torch.empty_like(u)
        for i, k in self.levels:
            v[i] = u[i] @ k
        v = (v * self.scale[:, None]).view(-1)
        return torch.zeros_like(x).index_add_(0, self.cols, self.vals * v[self.rows])


@functools.lru_cache(maxsize=1)
def _mask_ids(da):
    return _dev(da.boundary(), np.int64)


def _masked(A, ids, masked):
    def apply(x):
        if masked == 1:
            x = x.clone()
            x[ids] = 0.0
        y = A(x)
        if masked:
            y[ids] = 0.0
        return y
    return apply


def _cg(A, b, iters):
    x, r = torch.zeros_like(b), b.clone()
    p, rr = r.clone(), r @ r
    for _ in range(iters):
        ap = A(p)
        a = rr / (p @ ap)
        x += a * p
        r -= a * ap
        new = r @ r
        p = r + (new / rr) * p
        rr = new
    return x


def _bicgstab(A, b, iters):
    x, r = torch.zeros_like(b), b.clone()
    rh, p, v = r.clone(), torch.zeros_like(b), torch.zeros_like(b)
    rho, rho0, alpha, om = r @ r, 1.0, 1.0, 1.0
    for _ in range(iters):
        p = r + (rho / rho0) * (alpha / om) * (p - om * v)
        v = A(p)
        alpha = rho / (rh @ v)
        s = r - alpha * v
        t = A(s)
        om = (t @ s) / (t @ t)
        x += alpha * p + om * s
        r = s - om * t
        rho0, rho = rho, rh @ r
    return x


def exact(case, seed):
    kind = case["kind"]
    if case.get("points", 0) > 500000 or (kind == "cg" and case.get("level", 0) >= 9 and case["p"] == 2):
        return None  # the traversal's tables, or the products of the large solve, take too long
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)

    def operator(da, conforming, op="stiffness"):
        return _Conforming(da, op) if conforming else _Reference(da, op)

    if kind == "matvec":
        da = _da(case)
        shape = (da.n_nodes,) if case["nrhs"] == 1 else (da.n_nodes, case["nrhs"])
        x = _rand(shape, gen, DTYPE[case["dtype"]]).double()
        A = _masked(operator(da, case["conforming"], case["op"]), _mask_ids(da), case["masked"])
        if case["nrhs"] == 1:
            return A(x)
        return torch.stack([A(x[:, q].contiguous()) for q in range(case["nrhs"])], 1)
    if kind == "cg":
        da = _da(case)
        return _cg(_masked(operator(da, case["conforming"]), _mask_ids(da), 1), _rhs(da, gen), case["iters"])
    if kind == "bicgstab":
        da = _da(dict(case, dim=4))
        mats, ids = _captured(da)
        ids = _dev(ids, np.int64)
        b = _rand(da.n_nodes, gen)
        b[ids] = 0.0
        return _bicgstab(_masked(_Conforming(da, mats=mats), ids, 1), b, case["iters"])
    if kind == "cgbatch":
        das = _pool("serve", case["meshes"], case["lo"], case["hi"], case["mesh_seed"])
        bs = [_rhs(da, gen) for da in das]
        return [_cg(_masked(operator(da, True), _mask_ids(da), 1), b, case["iters"]) for da, b in zip(das, bs)]
    das = _pool("batch", case["trees"], case["lo"], case["hi"], case["mesh_seed"])
    out = []
    xs = [_rand((case["nrhs"], da.n_nodes), gen, DTYPE[case["dtype"]]) for da in das]
    for da, x in zip(das, xs):
        A = _Reference(da, "stiffness")
        out.append(torch.stack([A(x[q].double()) for q in range(case["nrhs"])]))
    return out
