"""The work a program has this library do, as cases that can be timed and compared.

Every case goes through the package's public classes (the solver classes on a ``Domain`` with
``Variable`` fields, ``SwEnsemble``, ``ServingEngine``), on the synthetic meshes and initial
states of the repository's benchmark and tests. A case is a dict of plain values:

* ``path``   which solver;
* ``nx, ny`` (2D) or ``n`` (3D): the mesh, 2 nx ny jittered triangles or 6 n^3 Kuhn tetrahedra;
* ``mode``   ``run`` (the solver's device-resident loop) or ``steps`` (a driver's own loop over
  ``stepper`` / ``compute_fluxes`` / ``compute_new_val``);
* ``steps``, ``order`` and the options of that solver.

``prepare`` makes the mesh (kept per size, as a program keeps it over many runs), the fields from
the seed and the solver; ``run`` resets the fields to the initial state and makes one call;
``exact`` computes the same in plain float64 torch, with another order of the sums.
"""
import copy
import functools
import math

import numpy as np
import torch

GRAV, GAMMA = 9.81, 1.4
WALLS = {"in": "nonslip", "out": "nonslip", "upper": "nonslip", "bottom": "nonslip"}
HOT_COLD = {"in": "dirichlet", "out": "dirichlet", "upper": "neumann", "bottom": "neumann"}


def listed():
    return [
        # a Gaussian blob advected over 80k triangles: 100 short, dependent steps
        {"name": "advection-run-80k", "path": "advection", "nx": 200, "ny": 200, "order": 1, "steps": 100,
         "mode": "run"},
        # second-order transport on a tetrahedral mesh, driven step by step
        {"name": "advection-3d-steps-197k", "path": "advection", "n": 32, "order": 2, "steps": 4, "mode": "steps"},
        # the dam break with MUSCL + Rusanov at production size: the solver's own loop
        {"name": "sw-rusanov-run-1M", "path": "sw", "flux": "rusanov", "nx": 708, "ny": 708, "order": 2, "steps": 10,
         "mode": "run"},
        # the same on the smallest mesh of an ensemble study: latency and launches
        {"name": "sw-rusanov-run-5k", "path": "sw", "flux": "rusanov", "nx": 61, "ny": 43, "order": 2, "steps": 30,
         "mode": "run"},
        # the default flux of ShallowWaterSolver, second order
        {"name": "sw-srnh-run-200k", "path": "sw", "flux": "srnh", "nx": 320, "ny": 313, "order": 2, "steps": 10,
         "mode": "run", "mann": 0.0},
        # the reference's own call sequence with friction on a mesh of test size
        {"name": "sw-srnh-steps-1k", "path": "sw", "flux": "srnh", "nx": 25, "ny": 23, "order": 1, "steps": 4,
         "mode": "steps", "mann": 0.02},
        # a Sod tube on 1.6M tetrahedra
        {"name": "euler-run-1.6M", "path": "euler", "n": 64, "steps": 10, "mode": "run"},
        # the same with dt read back each step, on a mesh of test size
        {"name": "euler-steps-8k", "path": "euler", "n": 11, "steps": 4, "mode": "steps"},
        # explicit advection-diffusion with the diamond gradient, second-order convection
        {"name": "advdiff-steps-100k", "path": "advdiff", "nx": 224, "ny": 223, "order": 2, "steps": 4,
         "mode": "steps"},
        # a stationary diffusion system (matrix kept, another right-hand side on each call)
        {"name": "solve-13k", "path": "solve", "nx": 80, "ny": 80},
        # uneven dam breaks advanced together from one captured graph, mixed precision
        {"name": "ensemble-24", "path": "ensemble", "count": 24, "lo": 5000, "hi": 60000, "steps": 30, "mesh": 1},
        # implicit advection-diffusion requests served together: admission, 20 steps, results
        {"name": "serving-8", "path": "serving", "count": 8, "lo": 10000, "hi": 60000, "steps": 20, "mesh": 2},
    ]


def draw(rng):
    """One more case: the path, then sizes spread over the logarithm of its range."""
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def rect(lo, hi):  # cells -> (nx, ny) with an aspect ratio of 1 to 4
        c, aspect = size(lo, hi), rng.uniform(1., 4.)
        ny = max(3, int(round(math.sqrt(c / (2. * aspect)))))
        return {"nx": max(3, int(round(c / (2. * ny)))), "ny": ny}

    path = rng.choice(["advection", "advection", "sw", "sw", "sw", "euler", "euler", "advdiff", "solve", "ensemble",
                       "serving"])
    mode = rng.choice(["run", "steps"])
    if path == "advection":
        shape = rect(1000, 200000) if rng.random() < .5 else {"n": size(5, 30)}
        order = rng.choice([1, 2])
        return dict(shape, path=path, order=order, steps=rng.randint(20, 80) if mode == "run" else rng.randint(2, 6),
                    mode=mode)
    if path == "sw":
        flux = rng.choice(["rusanov", "srnh"])
        shape = rect(1000, 800000 if flux == "rusanov" else 200000)
        c = dict(shape, path=path, flux=flux, order=rng.choice([1, 2]), mode=mode,
                 steps=rng.randint(5, 20) if mode == "run" else rng.randint(2, 5))
        if flux == "srnh":
            c["mann"] = rng.choice([0.0, 0.0, 0.02])
        return c
    if path == "euler":
        return {"path": path, "n": size(6, 56), "mode": mode,
                "steps": rng.randint(5, 20) if mode == "run" else rng.randint(2, 5)}
    if path == "advdiff":
        shape = rect(1000, 100000) if rng.random() < .6 else {"n": size(5, 24)}
        return dict(shape, path=path, order=rng.choice([1, 2]), steps=rng.randint(2, 5), mode="steps")
    if path == "solve":  # up to the size that the solver's default options converge for
        n = size(22, 80)
        return dict({"nx": n, "ny": n + rng.randint(0, 2)} if rng.random() < .7 else {"n": size(5, 14)}, path=path)
    if path == "ensemble":
        return {"path": path, "count": rng.randint(4, 24), "lo": 5000, "hi": size(10000, 60000),
                "steps": 6 * rng.randint(1, 5), "mesh": rng.randint(10, 10000)}
    return {"path": path, "count": rng.randint(2, 8), "lo": 10000, "hi": size(12000, 60000),
            "steps": rng.randint(5, 20), "mesh": rng.randint(10, 10000)}


# --- meshes and initial states -------------------------------------------------------------------


@functools.lru_cache(maxsize=None)
def _mesh(path, nx, ny, n):
    """A Domain of one size; its jitter comes from the size. The paths that hang tables or boundary
    values of their own on a Domain have one each."""
    from manapy_amd import Domain, jittered_triangles, kuhn_tetrahedra
    if n:
        return Domain(3, mesh=kuhn_tetrahedra(n, 1., 0.08, n))
    length = 100. if path == "sw" else 1.
    return Domain(2, mesh=jittered_triangles(nx, ny, length, length * ny / nx, 0.1, nx + ny))


def _domain(c):
    return _mesh(c["path"], c.get("nx", 0), c.get("ny", 0), c.get("n", 0))


@functools.lru_cache(maxsize=None)
def _instances(path, count, lo, hi, key):
    """``count`` meshes of lo to hi triangles, log-uniform, with aspect ratios of 1 to 4."""
    from manapy_amd import Domain, jittered_triangles
    rng = np.random.default_rng(key)
    out = []
    for _ in range(count):
        cells = math.exp(rng.uniform(math.log(lo), math.log(hi)))
        aspect = rng.uniform(1., 4.)
        ny = max(2, int(round(math.sqrt(cells / (2. * aspect)))))
        nx = max(2, int(round(aspect * ny)))
        ly = 100. if path == "ensemble" else 1.
        lx = ly * nx / ny if path == "ensemble" else 1.
        out.append((Domain(2, mesh=jittered_triangles(nx, ny, lx, ly, 0.1, int(rng.integers(1 << 30)))), lx, ly))
    return out


def _bumps(center, count, rng, lx, ly):
    """Gaussian bumps: amplitude 0 to 0.3, width 2 to 8."""
    z = np.zeros(len(center))
    for _ in range(count):
        a, w, x, y = rng.uniform(0., .3), rng.uniform(2., 8.), rng.uniform(0., lx), rng.uniform(0., ly)
        z += a * np.exp(-((center[:, 0] - x) ** 2 + (center[:, 1] - y) ** 2) / (w * w))
    return z


def _dam(center, lx, ly, rng, bumps):
    h = np.where(center[:, 0] < rng.uniform(.3, .7) * lx, 2., 1.)
    return h, np.zeros(len(h)), np.zeros(len(h)), _bumps(center, bumps, rng, lx, ly)


def _blob(center, dim, rng, s=0.005):
    return np.exp(-sum((center[:, k] - rng.uniform(.25, .75)) ** 2 for k in range(dim)) / s)


def _fields(c, seed):
    """The seeded inputs of a single-mesh case, as numpy arrays in the mesh's own numbering."""
    rng = np.random.default_rng(seed)
    d = _domain(c)
    cc, dim = d.cells.center, int(d.dim)
    if c["path"] in ("advection", "advdiff"):
        # a smooth, sheared velocity given on the faces; the cells take the mean over their faces
        a, s = rng.uniform(.3, 1.2), rng.uniform(.1, .4)
        fc = d.faces.center
        uf = math.cos(a) + s * fc[:, 1]
        vf = math.sin(a) - s * fc[:, 0]
        wf = np.full(len(fc), rng.uniform(.2, .6) if dim == 3 else 0.)
        f = {"u": _blob(cc, dim, rng, 0.005 if dim == 2 else 0.02), "uf": uf, "vf": vf, "wf": wf}
        if c["path"] == "advdiff":
            f["D"] = math.exp(rng.uniform(math.log(1e-3), math.log(1e-1)))
            f["left"], f["right"] = rng.uniform(.5, 1.), rng.uniform(0., .5)
        return f
    if c["path"] == "sw":
        h, hu, hv, z = _dam(cc, 100., 100. * c["ny"] / c["nx"], rng, 8)
        return {"h": h, "hu": hu, "hv": hv, "Z": z, "hc": .1 * h}
    if c["path"] == "euler":
        x, p = rng.uniform(.4, .6), rng.uniform(.08, .2)
        left = cc[:, 0] < x
        U = np.zeros((6, len(cc)))
        U[0], U[1] = np.where(left, 1., .125), np.where(left, 1., p)
        U[5] = U[1] / (GAMMA - 1.)
        return {"U": U}
    if c["path"] == "solve":
        return {"rhs": sum(rng.uniform(-40., 40.) * _blob(cc, dim, rng, .02) for _ in range(4))}
    raise ValueError(c["path"])


def _requests(c, seed):
    """Seeded request data: mesh, initial field, diffusivity."""
    rng = np.random.default_rng(seed)
    out = []
    for d, _, _ in _instances(c["path"], c["count"], c["lo"], c["hi"], c["mesh"]):
        out.append((d, _blob(d.cells.center, 2, rng), math.exp(rng.uniform(math.log(1e-3), math.log(1e-1)))))
    return out


def _states(c, seed):
    rng = np.random.default_rng(seed)
    return [_dam(d.cells.center, lx, ly, rng, int(rng.integers(1, 11)))
            for d, lx, ly in _instances(c["path"], c["count"], c["lo"], c["hi"], c["mesh"])]


# --- the calls -------------------------------------------------------------------------------------


def prepare(case, seed):
    from manapy_amd import (AdvectionDiffusionSolver, AdvectionSolver, EulerSolver3D, HIPKrylovSolver,
                            ShallowWaterSolver, Struct, Variable)
    c = case
    p = c["path"]
    if p == "ensemble":
        from manapy_amd.ensemble import SwEnsemble
        e = SwEnsemble([d for d, _, _ in _instances(p, c["count"], c["lo"], c["hi"], c["mesh"])], _states(c, seed),
                       grav=GRAV, cfl=.8, order=2)
        return {"case": c, "ens": e, "state0": e.state.clone(), "rings0": e.rings.clone()}
    if p == "serving":
        from manapy_amd.serving import AdvDiffRequest, ServingEngine
        # requests whose host tables are made (what the engine's preparation threads do on arrival)
        reqs = [AdvDiffRequest(i, d, u0, velocity=(1., .5), D=D, nsteps=c["steps"]).prepare()
                for i, (d, u0, D) in enumerate(_requests(c, seed))]
        return {"case": c, "engine": ServingEngine(max_cells=1 << 20, max_inst=64), "requests": reqs}
    d, f = _domain(c), _fields(c, seed)
    dev = lambda a: torch.as_tensor(a, dtype=torch.float64, device="cuda")  # noqa: E731
    s = {"case": c}
    if p == "advection" or p == "advdiff":
        if p == "advection":
            var = Variable(domain=d)
        else:
            var = Variable(domain=d, BC=HOT_COLD, values={"in": f["left"], "out": f["right"]})
        vel = [Variable(domain=d) for _ in range(int(d.dim))]
        for v, k in zip(vel, ("uf", "vf", "wf")):
            v.face[:] = dev(f[k])
            v.interpolate_facetocell()
        D = f.get("D", 0.)
        conf = Struct(order=c["order"], cfl=.4, Dxx=D, Dyy=D, Dzz=D if int(d.dim) == 3 else 0.) if p == "advdiff" \
            else Struct(order=c["order"], cfl=.4)
        s["solver"] = (AdvectionDiffusionSolver if p == "advdiff" else AdvectionSolver)(var, vel=tuple(vel), conf=conf)
        s["reset"] = [(var.cell, dev(f["u"]))]
    elif p == "sw":
        h, hu, hv = Variable(domain=d), Variable(domain=d, BC=WALLS), Variable(domain=d, BC=WALLS)
        hc, Z = Variable(domain=d), Variable(domain=d)
        conf = dict(order=c["order"], cfl=.8, flux=c["flux"])
        if c["flux"] == "srnh":
            conf["Mann"] = c["mann"]
        s["solver"] = ShallowWaterSolver(h=h, hvel=(hu, hv), hc=hc, Z=Z, conf=Struct(**conf))
        Z.cell[:] = dev(f["Z"])
        s["reset"] = [(h.cell, dev(f["h"])), (hu.cell, dev(f["hu"])), (hv.cell, dev(f["hv"])), (hc.cell, dev(f["hc"]))]
    elif p == "euler":
        s["solver"] = EulerSolver3D(d, f["U"], cfl=.8)
        s["reset"] = [(s["solver"].U, s["solver"].U.clone())]
    else:
        var = Variable(domain=d, BC=_solve_bc(d), values={"in": 1., "out": 2.})
        s["solver"] = HIPKrylovSolver(domain=d, var=var)
        s["rhs"] = dev(f["rhs"])
        s["reset"] = [(var.cell, torch.zeros_like(var.cell))]
    return s


def _solve_bc(d):
    return dict(HOT_COLD, front="neumann", back="neumann") if int(d.dim) == 3 else HOT_COLD


def run(state):
    c = state["case"]
    p = c["path"]
    if p == "ensemble":
        e = state["ens"]
        e.state.copy_(state["state0"])
        e.rings.copy_(state["rings0"])
        e.step_index = 0
        e.run_graph(c["steps"], chunk=c["steps"])
        return {"state": e.state, "time": e.rings[:, 3]}
    if p == "serving":
        done = state["engine"].run([copy.copy(r) for r in state["requests"]])
        return [r.result for r in sorted(done, key=lambda r: r.rid)]
    for field, start in state["reset"]:
        field.copy_(start)
    sol = state["solver"]
    if p == "solve":
        sol(state["rhs"])
        return {"x": sol.var.cell}
    if c["mode"] == "run":
        t = sol.run(c["steps"])
    elif p == "euler":
        t = 0.
        for _ in range(c["steps"]):
            t += sol.step()
    else:
        t = 0.
        for _ in range(c["steps"]):
            t += sol.stepper()
            sol.compute_fluxes()
            sol.compute_new_val()
    out = {"time": float(t)}
    if p == "euler":
        out["U"] = sol.U
    elif p == "sw":
        out.update(h=sol.h.cell, hu=sol.hu.cell, hv=sol.hv.cell)
        if c["flux"] == "srnh":
            out["hc"] = sol.hc.cell
    else:
        out["u"] = sol.var.cell
    return out


# --- what the work needs at least, and how close results have to be ---------------------------------


def _cells(c):
    if "count" in c:
        return int(sum(int(d.nbcells) for d, _, _ in _instances(c["path"], c["count"], c["lo"], c["hi"], c["mesh"])))
    return 6 * c["n"] ** 3 if c.get("n") else 2 * c["nx"] * c["ny"]


def work(case):
    """Bytes of one pass with every field and every geometry array that a step needs read once and
    every new field written once, in the width the path keeps it in; operations counted in the formulas."""
    c = case
    cells, p = _cells(c), c["path"]
    dim = 3 if c.get("n") else 2
    faces = (2. if dim == 3 else 1.5) * cells
    steps = c.get("steps", 1)
    slots = 4 if dim == 3 else 3
    order2 = c.get("order") == 2
    # a face: its two cells, normal and measure; with MUSCL its centre too
    face = 8 + 8 * dim + 8 + (8 * dim if order2 else 0)
    # a cell: its faces, volume; with MUSCL its centre and the stencil of its vertex neighbours
    sten = (70 if dim == 3 else 13) * 4
    cell = 4 * slots + 8 + (8 * dim + sten if order2 else 0)
    mesh = face * faces + cell * cells
    if p == "advection":
        b = mesh + 8 * dim * (faces + cells) + 16 * cells
        fl = cells * (slots * 12 + ((70 if dim == 3 else 13) * (18 if dim == 3 else 11) + 60 if order2 else 0))
    elif p == "advdiff":
        nodes = cells / (6. if dim == 3 else 2.)
        node_w = 12 * (4 if dim == 3 else 3) * cells + 4 * nodes
        diamond = (4 * dim + 8 * (2 * dim if dim == 3 else 8) + 8) * faces
        b = mesh + 8 * dim * (faces + cells) + 16 * cells + node_w + diamond
        fl = cells * (slots * 50 + ((70 if dim == 3 else 13) * 18 if order2 else 0))
    elif p == "sw":
        n = 5 if c["flux"] == "srnh" else 3
        b = mesh + 8 * (2 * n + 1) * cells
        fl = cells * (slots * (600 if n == 5 else 90) + (13 * 20 if order2 else 0))
    elif p == "euler":
        b = mesh + 96 * cells
        fl = cells * slots * 110
    elif p == "ensemble":
        b = (2 * 32 + 16 * 3 + 8 * 3 + 4 * 3 + 8 + 2 * 13) * cells
        fl = cells * (3 * 90 + 13 * 20)
    elif p == "solve":
        # the matrix (a column and a value an entry), the right-hand side and the solution
        b, fl = ((110 if dim == 3 else 14) * 12 + 24) * cells, 2. * (110 if dim == 3 else 14) * cells
    else:
        b, fl = (14 * 12 + 24 + 112) * cells, 2. * 14 * cells + 40. * cells
    return {"bytes": float(b * steps), "flops": float(fl * steps)}


def tolerance(case):
    """About four times what the path differs from the same in 64 bits with its sums in another
    order: rounding for the float64 paths; float32 for the ensemble's fluxes; the solver's stop at a
    relative residual of 1e-10 for the linear systems."""
    p = case["path"]
    if p == "ensemble":
        return {"rel": 1.6e-7, "max": 2e-6}
    if p == "solve":
        return {"rel": 3.5e-8, "max": 1e-7}
    if p == "serving":
        return {"rel": 3e-9, "max": 1e-8}
    return {"rel": 2e-13, "max": 1e-11}


# --- the same in plain float64 torch ------------------------------------------------------------------


class _Geo(object):
    """A mesh's arrays as torch tensors (its geometry and connectivity are inputs)."""

    def __init__(self, d):
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.d, self.dim = d, int(d.dim)
        self.C, self.F = int(d.nbcells), int(d.nbfaces)
        f = lambda a: torch.as_tensor(np.ascontiguousarray(a, dtype=np.float64), device=self.dev)  # noqa: E731
        i = lambda a: torch.as_tensor(np.ascontiguousarray(a, dtype=np.int64), device=self.dev)  # noqa: E731
        self.i, self.f = i, f
        self.L, R = i(d.faces.cellid[:, 0]), i(d.faces.cellid[:, 1])
        self.inner = R >= 0
        self.R = torch.where(self.inner, R, self.L)
        self.n, self.mes = f(d.faces.normal[:, :3]), f(d.faces.mesure)
        self.fc, self.cc, self.vol = f(d.faces.center[:, :3]), f(d.cells.center[:, :3]), f(d.cells.volume)
        fid = np.asarray(d.cells.faceid)
        w = fid.shape[1] - 1
        self.fid = i(np.where(np.arange(w)[None, :] < fid[:, -1:], fid[:, :w], 0))
        self.fok = torch.as_tensor(np.arange(w)[None, :] < fid[:, -1:], device=self.dev)
        gc = np.zeros((self.F, 3))
        gc[:, :self.dim] = d.faces.ghostcenter[:, :self.dim]
        self.gc = f(gc)
        self.name = i(d.faces.name)

    def stencil(self):
        if not hasattr(self, "sten"):
            d, out = self.d, []
            for t in (d.cells.cellnid, d.cells.ghostnid):
                w = t.shape[1] - 1
                ok = np.arange(w)[None, :] < t[:, -1:]
                out.append((self.i(np.where(ok, t[:, :w], 0)), torch.as_tensor(ok, device=self.dev)))
            self.sten = out
        return self.sten

    def sum_faces(self, per_face):
        """sum over a cell's faces of per_face."""
        return (per_face[self.fid] * self.fok).sum(1)

    def scatter(self, flux):
        r = torch.zeros(self.C, dtype=torch.float64, device=self.dev)
        r.index_add_(0, self.L, -flux)
        return r.index_add_(0, self.R[self.inner], flux[self.inner])

    def gradient(self, w, ghost):
        """Least squares over the vertex neighbours and the ghosts of the boundary faces."""
        (cn, cok), (gn, gok) = self.stencil()
        dim = self.dim
        A = torch.zeros((self.C, dim, dim), dtype=torch.float64, device=self.dev)
        b = torch.zeros((self.C, dim), dtype=torch.float64, device=self.dev)
        for idx, ok, pts, val in ((cn, cok, self.cc, w), (gn, gok, self.gc, ghost)):
            for k in range(idx.shape[1]):
                r = (pts[idx[:, k], :dim] - self.cc[:, :dim]) * ok[:, k:k + 1]
                A += r[:, :, None] * r[:, None, :]
                b += r * (val[idx[:, k]] - w)[:, None]
        if dim == 2:
            det = A[:, 0, 0] * A[:, 1, 1] - A[:, 0, 1] ** 2
            return torch.stack([(A[:, 1, 1] * b[:, 0] - A[:, 0, 1] * b[:, 1]) / det,
                                (A[:, 0, 0] * b[:, 1] - A[:, 0, 1] * b[:, 0]) / det], 1)
        c0, c1, c2 = A[:, :, 0], A[:, :, 1], A[:, :, 2]
        det = (c0 * torch.linalg.cross(c1, c2)).sum(1)
        return torch.stack([(b * torch.linalg.cross(c1, c2)).sum(1), (b * torch.linalg.cross(c2, c0)).sum(1),
                            (b * torch.linalg.cross(c0, c1)).sum(1)], 1) / det[:, None]

    def limiter(self, w, ghost, g):
        """Barth-Jespersen."""
        eps = 1e-8 if self.dim == 2 else 1e-10
        lf = w[self.L]
        rf = torch.where(self.inner, w[self.R], ghost)
        hi = torch.maximum(lf, rf)[self.fid].masked_fill(~self.fok, -math.inf).max(1).values
        lo = torch.minimum(lf, rf)[self.fid].masked_fill(~self.fok, math.inf).min(1).values
        hi, lo = torch.maximum(hi, w), torch.minimum(lo, w)
        delta = (g[:, None, :] * (self.fc[self.fid] - self.cc[:, None, :])[:, :, :self.dim]).sum(2)
        room = torch.where(delta > 0, (hi - w)[:, None], (lo - w)[:, None])
        flat = (delta.abs() < eps) | ~self.fok
        psi = torch.where(flat, 1., (room / torch.where(flat, 1., delta)).clamp(max=1.))
        return psi.min(1).values.clamp(max=1.)

    def face_values(self, w, g, psi=None):
        """Both sides' reconstructed values at each face (the right one of an inner face)."""
        out = []
        for side in (self.L, self.R):
            inc = (g[side] * (self.fc - self.cc[side])[:, :self.dim]).sum(1)
            out.append(w[side] + (inc if psi is None else psi[side] * inc))
        return out


def _np(t):
    return t.cpu().numpy()


def _exact_transport(c, seed):
    d, f = _domain(c), _fields(c, seed)
    g = _Geo(d)
    u = g.f(f["u"])
    vf = torch.stack([g.f(f[k]) for k in ("uf", "vf", "wf")], 1)
    cnt = g.fok.sum(1)
    vc = torch.stack([g.sum_faces(vf[:, k]) / cnt for k in range(3)], 1)
    un = (vf * g.n).sum(1)
    lam = ((vc[:, None, :] * g.n[g.fid]).sum(2).abs() * g.fok).sum(1)
    diff = c["path"] == "advdiff"
    if diff:
        lam = lam + g.dim * f["D"] * g.sum_faces((g.n ** 2).sum(1)) / g.vol
        node = _node_weights(g)
    dt = float((.4 * g.vol / lam).min())
    t = 0.
    for _ in range(c["steps"]):
        t += dt
        ghost = u[g.L]
        if diff:
            for loc, val in (("in", f["left"]), ("out", f["right"])):
                ghost = ghost.masked_fill(g.name == {"in": 1, "out": 2}[loc], val)
        left, right = u[g.L], torch.where(g.inner, u[g.R], ghost)
        if c["order"] == 2:
            gr = g.gradient(u, ghost)
            lv, rv = g.face_values(u, gr, g.limiter(u, ghost, gr))
            left, right = lv, torch.where(g.inner, rv, ghost)
        rez = g.scatter(un * torch.where(un >= 0, left, right))
        if diff:
            q = f["D"] * (_face_gradient(g, u, ghost, node) * g.n[:, :g.dim]).sum(1)
            rez = rez - g.scatter(q)
        u = u + dt * rez / g.vol
    return {"time": t, "u": _np(u)}


def _node_weights(g):
    """(node, cell or face, weight) of the least-squares node interpolation, cells and ghosts apart."""
    d, nd = g.d, g.d.nodes
    den = nd.number + nd.lambda_x * nd.R_x + nd.lambda_y * nd.R_y
    if g.dim == 3:
        den = den + nd.lambda_z * nd.R_z
    out = []
    for table, pts in ((nd.cellid, d.cells.center), (nd.ghostid, d.faces.ghostcenter)):
        w = table.shape[1] - 1
        ok = np.arange(w)[None, :] < table[:, -1:]
        n, k = np.nonzero(ok)
        j = table[n, k].astype(np.int64)
        a = 1. + nd.lambda_x[n] * (pts[j, 0] - nd.vertex[n, 0]) + nd.lambda_y[n] * (pts[j, 1] - nd.vertex[n, 1])
        if g.dim == 3:
            a = a + nd.lambda_z[n] * (pts[j, 2] - nd.vertex[n, 2])
        out.append((n, j, a / den[n]))
    return out


def _face_nodes(g):
    fn = np.asarray(g.d.faces.nodeid)
    return fn[:, [0, 1]] if g.dim == 2 else fn[:, [0, 1, 2, 2]]


def _face_gradient(g, u, ghost, node):
    d = g.d
    if not hasattr(g, "fgrad"):
        g.fgrad = [(g.i(n), g.i(j), g.f(a)) for n, j, a in node] + [g.i(_face_nodes(g)), g.f(d.faces.airDiamond)] + \
            [g.f(x) for x in ((d.faces.f_1, d.faces.f_2, d.faces.f_3, d.faces.f_4) if g.dim == 2
                              else (d.faces.f_1, d.faces.f_2))]
    (n0, j0, a0), (n1, j1, a1), fn, air = g.fgrad[:4]
    fk = g.fgrad[4:]
    w = torch.zeros(int(d.nbnodes), dtype=torch.float64, device=g.dev)
    w.index_add_(0, n0, a0 * u[j0])
    w.index_add_(0, n1, a1 * ghost[j1])
    vl, vr = u[g.L], torch.where(g.inner, u[g.R], ghost)
    if g.dim == 2:
        v1, v2 = w[fn[:, 0]], w[fn[:, 1]]
        s = (v1 + vl)[:, None] * fk[0] + (vl + v2)[:, None] * fk[1] + (v2 + vr)[:, None] * fk[2] + \
            (vr + v1)[:, None] * fk[3]
        return torch.stack([s[:, 1], -s[:, 0]], 1) / (2. * air)[:, None]
    a, b, cc_, dd = (w[fn[:, k]] for k in range(4))
    return (fk[0] * (a - cc_)[:, None] + fk[1] * (b - dd)[:, None] + g.n * (vr - vl)[:, None]) / air[:, None]


def _sw_dt(g, h, hu, hv):
    un = (torch.stack([hu / h, hv / h], 1)[:, None, :] * g.n[g.fid][:, :, :2]).sum(2).abs()
    lam = ((un + (GRAV * h).sqrt()[:, None] * g.mes[g.fid]) * g.fok).sum(1)
    return float((.8 * g.vol / lam).min())


def _exact_rusanov(d, st, order, steps):
    g = _Geo(d)
    h, hu, hv, z = (g.f(a) for a in st)
    zg = g.gradient(z, z[g.L])
    zl, zr = g.face_values(z, zg) if order == 2 else (z[g.L], z[g.R])
    n0, n1 = g.n[:, 0], g.n[:, 1]
    t = 0.
    for _ in range(steps):
        dt = _sw_dt(g, h, hu, hv)
        t += dt
        sides = [[], []]
        for w, sgn in ((h + z, 1.), (hu, -1.), (hv, -1.)):
            if order == 2:
                ghost = sgn * w[g.L]
                gr = g.gradient(w, ghost)
                lv, rv = g.face_values(w, gr, g.limiter(w, ghost, gr))
            else:
                lv, rv = w[g.L], w[g.R]
            sides[0].append(lv)
            sides[1].append(torch.where(g.inner, rv, sgn * lv))
        zfl, zfr = zl, torch.where(g.inner, zr, zl)
        zs = torch.maximum(zfl, zfr)
        q, p, hs, vel, sp, src = [], [], [], [], [], []
        for (e, a, b), zf, own in zip(sides, (zfl, zfr), (g.L, g.R)):
            hf = (e - zf).clamp(min=0.)
            wet = hf > 1e-12
            safe = torch.where(wet, hf, 1.)
            uu, vv = torch.where(wet, a / safe, 0.), torch.where(wet, b / safe, 0.)
            s = (hf + zf - zs).clamp(min=0.)
            q.append(uu * n0 + vv * n1)
            p.append(.5 * GRAV * s * s)
            hs.append(s)
            vel.append((uu, vv))
            sp.append(q[-1].abs() / g.mes + (GRAV * s).sqrt())
            src.append(.5 * GRAV * (hf * hf - s * s) + GRAV * (hf + h[own]) * .5 * (zf - z[own]))
        s = torch.maximum(*sp) * g.mes
        new = []
        for k, w in enumerate((h, hu, hv)):
            if k == 0:
                fl = .5 * (hs[0] * q[0] + hs[1] * q[1]) - .5 * s * (hs[1] - hs[0])
                rez = g.scatter(fl)
            else:
                n = (n0, n1)[k - 1]
                m = [hs[i] * vel[i][k - 1] for i in (0, 1)]
                fl = .5 * (m[0] * q[0] + p[0] * n + m[1] * q[1] + p[1] * n) - .5 * s * (m[1] - m[0])
                rez = g.scatter(fl)
                rez.index_add_(0, g.L, -src[0] * n)
                rez.index_add_(0, g.R[g.inner], (src[1] * n)[g.inner])
            new.append(w + dt * rez / g.vol)
        h, hu, hv = new
    return t, _np(h), _np(hu), _np(hv)


def _srnh_flux(left, right, n0, n1, mes):
    """The SRNH flux of (hu, hv, h, hc, Z) on both sides of each face."""
    (hul, hvl, hl, hcl, zl), (hur, hvr, hr, hcr, zr) = left, right
    sl, sr = hl.sqrt(), hr.sqrt()
    mean = lambda a, b: (a / hl * sl + b / hr * sr) / (sl + sr)  # noqa: E731
    uh, vh, c = mean(hul, hur), mean(hvl, hvr), mean(hcl, hcr)
    u, v, h = (uh * n0 + vh * n1) / mes, (-uh * n1 + vh * n0) / mes, (hl + hr) / 2.
    ul, vl, ur, vr = ((a * x + b * y) / mes for a, b, x, y in
                      ((hul, hvl, n0, n1), (hul, hvl, -n1, n0), (hur, hvr, n0, n1), (hur, hvr, -n1, n0)))
    avg = [(hl + hr) / 2., (ul + ur) / 2., (vl + vr) / 2., (hcl + hcr) / 2.]
    dif = [hr - hl, ur - ul, vr - vl, hcr - hcl, zr - zl]
    Q = -(u * u + 3. * GRAV * h) / 9.
    th = torch.arccos(u * (18. * GRAV * h - 2. * u * u) / 54. / (-Q ** 3).sqrt())
    lam = [2. * (-Q).sqrt() * torch.cos((th + k * math.pi) / 3.) + 2. / 3. * u for k in (0., 2., 4.)]
    a1, a2, a3 = (x - u for x in lam)
    s1, s2, s3 = (torch.where(x.abs() < 1e-10, 0., x.sign()) for x in lam)
    s4 = torch.where(u.abs() < 1e-10, 0., u.sign())
    ss = GRAV * h
    G = [(ss - u * u + x) / y for x, y in
         ((lam[1] * lam[2], -a1 * a2 + a2 * a3 - a1 * a3 + a1 * a1),
          (lam[0] * lam[2], a1 * a2 + a2 * a3 - a1 * a3 - a2 * a2),
          (lam[0] * lam[1], a1 * a2 - a2 * a3 - a1 * a3 + a3 * a3))]
    sg = [-a1 * a2 + a2 * a3 - a1 * a3 + a1 * a1, a1 * a2 + a2 * a3 - a1 * a3 - a2 * a2,
          a1 * a2 - a2 * a3 - a1 * a3 + a3 * a3]
    sn = (s1, -s2, s3)
    pair = (a2 + a3, a1 + a3, a1 + a2)
    w = [sn[k] * (G[k] * dif[0] - pair[k] / sg[k] * dif[1] + ss / sg[k] * dif[4]) for k in range(3)]
    tot = w[0] + w[1] + w[2]
    cor = [tot, lam[0] * w[0] + lam[1] * w[1] + lam[2] * w[2], v * tot - v * s4 * dif[0] + s4 * dif[2],
           c * tot - c * s4 * dif[0] + s4 * dif[3]]
    hs, us, vs, cs = (x - y / 2. for x, y in zip(avg, cor))
    un, vn = (us * n0 - vs * n1) / mes, (us * n1 + vs * n0) / mes
    q = n0 * un + n1 * vn
    return [q, q * un / hs + .5 * GRAV * hs * hs * n0, q * vn / hs + .5 * GRAV * hs * hs * n1, q * cs / hs]


def _srnh_source(g, h, z, hg, zg):
    d = g.d
    if not hasattr(g, "src"):
        # the neighbour behind slot j as the scheme takes it: the j-th entry of the cell's neighbour list
        nb = np.asarray(d.cells.cellfid)[:, :3].astype(np.int64)
        g.src = (g.i(np.where(nb < 0, nb + g.C, nb)), g.f(d.cells.nf[:, :, :2]),
                 g.f(d.nodes.vertex[np.asarray(d.cells.nodeid)[:, 1], :2]))
    nb, ss, b = g.src
    fid = g.fid[:, :3]
    inner = g.name[fid] == 0
    hp, zp = torch.where(inner, h[nb], hg[fid]), torch.where(inner, z[nb], zg[fid])
    m = hp[:, :, None] * ss
    c1 = ((.5 * (h[:, None] + hp)) ** 2)[:, :, None] * ss
    c1, c2 = c1.sum(1)[:, 0], c1.sum(1)[:, 1]
    c3 = 3. * h
    a, e = m[:, :, 0], m[:, :, 1]
    x12, x02, x01 = (a[:, i] * e[:, j] - a[:, j] * e[:, i] for i, j in ((1, 2), (0, 2), (0, 1)))
    y = [c1 * e[:, k] - c2 * a[:, k] for k in range(3)]
    det = x12 - x02 + x01
    hh = [(c3 * x12 - y[2] + y[1]) / det, (y[2] - c3 * x02 - y[0]) / det, (-y[1] + y[0] + c3 * x01) / det]
    zz = [z + h - x for x in hh]
    n0 = torch.stack([g.cc[:, 1] - b[:, 1], -(g.cc[:, 0] - b[:, 0])], 1)
    n1, n2 = n0 - ss[:, 1], n0 + ss[:, 0]
    col = lambda t: t[:, None]  # noqa: E731
    s = col(.5 * hh[0]) * (col(zp[:, 0]) * ss[:, 0] + col(zz[1]) * n0 - col(zz[2]) * n2) + \
        col(.5 * hh[1]) * (col(zp[:, 1]) * ss[:, 1] - col(zz[0]) * n0 + col(zz[2]) * n1) + \
        col(.5 * hh[2]) * (col(zp[:, 2]) * ss[:, 2] + col(zz[0]) * n2 - col(zz[1]) * n1)
    return -GRAV * s[:, 0], -GRAV * s[:, 1]


def _exact_srnh(c, seed):
    g, f = _Geo(_domain(c)), _fields(c, seed)
    h, hu, hv, hc, z = (g.f(f[k]) for k in ("h", "hu", "hv", "hc", "Z"))
    n0, n1 = g.n[:, 0], g.n[:, 1]
    pick = lambda l, r: torch.where(g.inner, r, l)  # noqa: E731
    t = 0.
    for _ in range(c["steps"]):
        first = dt = _sw_dt(g, h, hu, hv)
        if c["mann"]:
            A = 1. + dt * GRAV * c["mann"] ** 2 * ((hu / h) ** 2 + (hv / h) ** 2).sqrt() / h ** (4. / 3.)
            hu, hv = hu / A, hv / A
            dt = _sw_dt(g, h, hu, hv)
        t += first if c["mode"] == "steps" else dt
        L = [hu[g.L], hv[g.L], h[g.L], hc[g.L], z[g.L]]
        gh = [-L[0], -L[1], L[2], L[3], L[4]]
        R = [w[g.R] for w in (hu, hv, h, hc, z)]
        if c["order"] == 2:
            gc = g.gradient(hc, gh[3])
            psi = g.limiter(hc, gh[3], gc)
            L[2], R[2] = g.face_values(h, g.gradient(h, gh[2]), psi)
            L[3], R[3] = g.face_values(hc, gc, psi)
        fl = _srnh_flux(L, [pick(a, b) for a, b in zip(gh, R)], n0, n1, g.mes)
        sx, sy = _srnh_source(g, h, z, gh[2], gh[4])
        h, hu, hv, hc = (w + dt * (g.scatter(x) + s) / g.vol
                         for w, x, s in zip((h, hu, hv, hc), fl, (0., sx, sy, 0.)))
    return {"time": t, "h": _np(h), "hu": _np(hu), "hv": _np(hv), "hc": _np(hc)}


def _exact_euler(c, seed):
    g = _Geo(_domain(c))
    rho, P, *m, E = (g.f(a) for a in _fields(c, seed)["U"])
    m = torch.stack(m, 1)
    n = g.n / g.mes[:, None]
    slip = (g.name >= 3) & (g.name <= 6)
    unit = g.n / (g.n ** 2).sum(1).sqrt()[:, None]
    t = 0.
    for _ in range(c["steps"]):
        snd = (GAMMA * (P / rho).abs()).sqrt()
        un = ((m / rho[:, None])[:, None, :] * g.n[g.fid]).sum(2).abs() / (g.n ** 2).sum(1).sqrt()[g.fid]
        dt = float((.8 * g.vol / ((un + snd[:, None]) * g.mes[g.fid] * g.fok).sum(1)).min())
        t += dt
        sides = []
        for own in (g.L, g.R):
            mm = m[own]
            if own is g.R:
                flip = mm - 2. * (mm * unit).sum(1)[:, None] * unit
                mm = torch.where((slip & ~g.inner)[:, None], flip, mm)
            r, p, e = rho[own], P[own], E[own]
            q = (mm * n).sum(1)
            cs = (GAMMA * p / r).sqrt()
            sides.append((r, mm, e, q, mm * (q / r)[:, None] + p[:, None] * n, q / r * (e + p),
                          torch.maximum((q / r - cs).abs(), (q / r + cs).abs())))
        (rl, ml, el, ql, fml, fel, sl), (rr, mr, er, qr, fmr, fer, sr) = sides
        s = torch.maximum(sl, sr)
        jump = lambda a, b, x, y: (.5 * (a + b) - .5 * s * (y - x)) * g.mes  # noqa: E731
        fr, fe = jump(ql, qr, rl, rr), jump(fel, fer, el, er)
        fm = [jump(fml[:, k], fmr[:, k], ml[:, k], mr[:, k]) for k in range(3)]
        rho = rho + dt * g.scatter(fr) / g.vol
        m = m + dt * torch.stack([g.scatter(x) for x in fm], 1) / g.vol[:, None]
        E = E + dt * g.scatter(fe) / g.vol
        P = (GAMMA - 1.) * (E - .5 * (m ** 2).sum(1) / rho)
    return {"time": t, "U": _np(torch.stack([rho, P, m[:, 0], m[:, 1], m[:, 2], E]))}


def _diamond_matrix(g, dirichlet):
    """(row, col, value) of the diamond diffusion operator and the lifting of the Dirichlet values
    {boundary tag: value}."""
    d = g.d
    cid, vol, name = np.asarray(d.faces.cellid), d.cells.volume, np.asarray(d.faces.name)
    p1, p2, p3, p4 = d.faces.param1, d.faces.param2, d.faces.param3, d.faces.param4
    fn = _face_nodes(g)
    par = np.stack([p4, p2], 1) if g.dim == 2 else np.stack([p1, p2, -p1, -p2], 1)
    on = np.asarray(d.nodes.oldname)
    fixed = np.isin(on, list(dirichlet))
    pin = np.zeros(len(on))
    for tag, val in dirichlet.items():
        pin[on == tag] = val
    # per node: the cells its value is made of (a ghost counts for its owner)
    (n0, c0, a0), (n1, f1, a1) = _node_weights(g)
    nn, cc, aa = np.concatenate([n0, n1]), np.concatenate([c0, cid[f1, 0]]), np.concatenate([a0, a1])
    o = np.argsort(nn, kind="stable")
    cc, aa = cc[o], aa[o]
    cnt = np.bincount(nn, minlength=len(on))
    start = np.cumsum(cnt) - cnt
    inner = np.nonzero(cid[:, 1] >= 0)[0]
    l, r = cid[inner, 0], cid[inner, 1]
    own = p1 if g.dim == 2 else -p3
    rows, cols, vals = [l, l, r, r], [l, r, l, r], [own[inner] / vol[l], p3[inner] / vol[l], -own[inner] / vol[r],
                                                   -p3[inner] / vol[r]]
    rhs = np.zeros(g.C)
    for k in range(fn.shape[1]):
        node, w = fn[inner, k], par[inner, k]
        pinned = fixed[node]
        np.add.at(rhs, l[pinned], -(pin[node] * w / vol[l])[pinned])
        np.add.at(rhs, r[pinned], (pin[node] * w / vol[r])[pinned])
        free = np.nonzero(~pinned)[0]
        rep = cnt[node[free]]
        e = np.repeat(free, rep)
        at = np.repeat(start[node[free]], rep) + np.arange(len(e)) - np.repeat(np.cumsum(rep) - rep, rep)
        for side, sgn in ((l, 1.), (r, -1.)):
            rows.append(side[e])
            cols.append(cc[at])
            vals.append(sgn * aa[at] * w[e] / vol[side[e]])
    bf = np.nonzero(np.isin(name, list(dirichlet)) & (cid[:, 1] < 0))[0]
    b = cid[bf, 0]
    rows.append(b)
    cols.append(b)
    vals.append((own[bf] - p3[bf]) / vol[b])
    for k in range(fn.shape[1]):
        np.add.at(rhs, b, -pin[fn[bf, k]] * par[bf, k] / vol[b])
    value = np.zeros(len(name))
    for tag, val in dirichlet.items():
        value[name == tag] = val
    np.add.at(rhs, b, -2. * p3[bf] / vol[b] * value[bf])
    return g.i(np.concatenate(rows)), g.i(np.concatenate(cols)), g.f(np.concatenate(vals)), g.f(rhs)


def _solve(op, diag, b, x, tol=1e-14, most=40):
    """BiCGStab with Jacobi scaling, restarted from the true residual until it stops falling."""
    inv, best = 1. / diag, math.inf
    for _ in range(most):
        r = b - op(x)
        rn = float(r.norm() / b.norm())
        if rn <= tol or rn > .5 * best:
            break
        best = rn
        d, rh, r0 = torch.zeros_like(b), r.clone(), float(r.norm())
        p, rho = r.clone(), torch.dot(r, r)
        for it in range(20000):
            y = inv * p
            v = op(y)
            al = rho / torch.dot(rh, v)
            s = r - al * v
            z = inv * s
            t = op(z)
            om = torch.dot(t, s) / torch.dot(t, t)
            d += al * y + om * z
            r = s - om * t
            new = torch.dot(rh, r)
            p = r + new / rho * al / om * (p - om * v)
            rho = new
            if it % 10 == 9 and not float(r.norm()) > 1e-7 * r0:
                break
        if not bool(torch.isfinite(d).all()):
            break
        x = x + d
    return x


def _rows_of(row, col, val, size):
    """The matrix as padded rows: y = (vals * x[cols]).sum(1)."""
    key = row * size + col
    key, inv = torch.unique(key, return_inverse=True)
    v = torch.zeros(len(key), dtype=torch.float64, device=val.device).index_add_(0, inv, val)
    r, c = key // size, key % size
    cnt = torch.bincount(r, minlength=size)
    slot = torch.arange(len(r), device=r.device) - (torch.cumsum(cnt, 0) - cnt)[r]
    cols = torch.zeros((size, int(cnt.max())), dtype=torch.int64, device=r.device)
    vals = torch.zeros(cols.shape, dtype=torch.float64, device=r.device)
    cols[r, slot], vals[r, slot] = c, v
    diag = torch.zeros(size, dtype=torch.float64, device=r.device).index_add_(0, r[r == c], v[r == c])
    return cols, vals, diag


def _exact_solve(c, seed):
    g = _Geo(_domain(c))
    row, col, val, rhs0 = _diamond_matrix(g, {1: 1., 2: 2.})
    cols, vals, diag = _rows_of(row, col, val, g.C)
    b = rhs0 + g.f(_fields(c, seed)["rhs"])
    x = _solve(lambda x: (vals * x[cols]).sum(1), diag, b, torch.zeros_like(b))
    return {"x": _np(x)}


def _exact_serving(c, seed):
    out = []
    for d, u0, D in _requests(c, seed):
        g = _Geo(d)
        cols, vals, diag = _rows_of(*_diamond_matrix(g, {})[:3], g.C)
        u = g.f(u0)
        un = g.n[:, 0] + .5 * g.n[:, 1]
        dt = float((.8 * g.vol / g.sum_faces(un.abs())).min())
        tau = -dt * D
        for _ in range(c["steps"]):
            b = u + dt * g.scatter(un * torch.where(un >= 0, u[g.L], u[g.R])) / g.vol
            u = _solve(lambda x: x + tau * (vals * x[cols]).sum(1), 1. + tau * diag, b, b.clone())
        out.append(_np(u))
    return out


def _exact_ensemble(c, seed):
    """In the ensemble's own layout: instances at multiples of 64 cells, cells along the curve."""
    from manapy_amd.renumber import renumbered
    rows, times = [], []
    for (d, _, _), st in zip(_instances(c["path"], c["count"], c["lo"], c["hi"], c["mesh"]), _states(c, seed)):
        t, h, hu, hv = _exact_rusanov(d, st, 2, c["steps"])
        a = np.stack([h, hu, hv, st[3]], 1)[renumbered(d).perm]
        rows.append(np.concatenate([a, np.zeros((-len(a) % 64, 4))]))
        times.append(t)
    return {"state": np.concatenate(rows), "time": np.array(times)}


def exact(case, seed):
    c, p = case, case["path"]
    if p in ("advection", "advdiff"):
        return _exact_transport(c, seed)
    if p == "sw" and c["flux"] == "srnh":
        return _exact_srnh(c, seed)
    if p == "sw":
        f = _fields(c, seed)
        t, h, hu, hv = _exact_rusanov(_domain(c), [f[k] for k in ("h", "hu", "hv", "Z")], c["order"], c["steps"])
        return {"time": t, "h": h, "hu": hu, "hv": hv}
    if p == "euler":
        return _exact_euler(c, seed)
    return {"solve": _exact_solve, "serving": _exact_serving, "ensemble": _exact_ensemble}[p](c, seed)
