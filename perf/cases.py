"""The work that is timed: the calls a program makes on this library, over the
range of grids, precisions and options that it makes them for.

    listed()             the named cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  what the program holds before the call, on the GPU
    run(state)           one pass through the public entry points
    work(case)           the bytes and operations a pass cannot do without
    exact(case, seed)    the outputs in 64 bits, in plain torch

Kinds of case:
    reinit     LevelSet.reinitialize_* on a device array: grids of one tree on
               [0, box]^dim, refined where |phi0| <= 1.2 diag(cell)
    host       the same on an array in host memory (a PETSc Vec's array)
    batch      TreeBatch.reinitialize_2nd_order over many small quadtrees
    advect     LevelSet.advect_in_normal_direction with its CFL time step
    curvature  normals, mean curvature, 3x3x3 samples and the learned blend
    train      curvature.train on stencils of circles
    regrid     DeviceGrid, sampling and a short reinitialization: one step of
               a loop that rebuilds its grid around a moving interface
"""
import functools
import math
import os
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import torch

import casl_p4est_amd as C
from casl_p4est_amd import curvature as CV
from casl_p4est_amd import levelset as ls

# my_p4est_level_set_t's entry points by the order of accuracy: (method, space, pseudo-time)
ORDERS = {
    "2nd": ("reinitialize_2nd_order", 2, 2),
    "1st_time": ("reinitialize_1st_order_time_2nd_order_space", 2, 1),
    "1st_space": ("reinitialize_2nd_order_time_1st_order_space", 1, 2),
    "1st": ("reinitialize_1st_order", 1, 1),
}


def _reinit(name, shape, lmin, lmax, precision, iters, items=0, box=1.0, order="2nd", graph=False):
    return dict(name=name, kind="reinit", dim=2 if shape == "star" else 3, shape=shape, items=items, lmin=lmin,
                lmax=lmax, box=box, precision=precision, order=order, iters=iters, graph=graph)


def _grid3(name, kind, lmax, items, iters=0, lmin=4):
    return dict(name=name, kind=kind, dim=3, shape="spheres", items=items, lmin=lmin, lmax=lmax, box=1.0, iters=iters)


def listed():
    return [
        # the smallest grid in use, a 2D contour in full precision: launches and latency
        _reinit("star2d_fp64", "star", 4, 9, "fp64", 20),
        # a fine 2D contour, mixed precision, replayed from a recorded graph as a time-stepping loop would
        _reinit("star2d_fine_mixed_graph", "star", 4, 12, "mixed", 20, graph=True),
        # a small 3D grid, the share one rank of a CPU run holds, first order in time
        _reinit("spheres3d_small_fp64", "spheres", 3, 6, "fp64", 10, items=12, order="1st_time"),
        # an ordinary 3D grid on a box whose edge is not a power of two
        _reinit("spheres3d_box3_fp64", "spheres", 4, 8, "fp64", 20, items=64, box=3.0),
        # many hanging nodes: a triply periodic surface that fills the box, full precision
        _reinit("gyroid3d_fp64", "gyroid", 5, 9, "fp64", 10),
        # the largest: 64 spheres at level 10, mixed precision, 50 iterations
        _reinit("spheres3d_large_mixed", "spheres", 5, 10, "mixed", 50, items=64),
        # an MPI code's own array in host memory, in and out on each call
        dict(_grid3("spheres3d_host_fp64", "host", 9, 64, iters=10), precision="fp64", order="2nd"),
        # many independent quadtrees in one launch
        dict(name="trees2d_batch_mixed", kind="batch", trees=512, lmin=3, lmax_lo=6, lmax_hi=9, precision="mixed",
             iters=20),
        # an interface moved along its normal by a velocity field
        _grid3("advect3d", "advect", 9, 64),
        # curvature of the interface, numerical and learned
        _grid3("curvature3d", "curvature", 9, 64),
        # one epoch of the 2D curvature network
        dict(name="train2d", kind="train", samples=131072, batch=16384),
        # a moving interface's grid rebuilt on the GPU
        dict(_grid3("regrid3d_mixed", "regrid", 9, 64, iters=5), precision="mixed"),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    u = rng.random()
    if u < 0.25:  # 2D contours
        return _drop_name(_reinit("", "star", rng.randint(3, 5), rng.randint(7, 13),
                                  rng.choice(["fp64", "mixed"]), log_int(5, 50),
                                  box=rng.choice([1.0, 1.0, 2.0, 3.0, 2.5]),
                                  order=rng.choice(["2nd", "2nd", "1st_time", "1st_space", "1st"]),
                                  graph=rng.random() < 0.25))
    if u < 0.60:  # 3D surfaces
        shape = rng.choice(["spheres", "spheres", "gyroid"])
        items = log_int(4, 64) if shape == "spheres" else 0
        c = _reinit("", shape, rng.randint(3, 5), rng.randint(6, 10 if shape == "spheres" else 9),
                    rng.choice(["fp64", "mixed"]), log_int(5, 50), items=items,
                    box=rng.choice([1.0, 1.0, 2.0, 3.0]),
                    order=rng.choice(["2nd", "2nd", "1st_time", "1st_space", "1st"]), graph=rng.random() < 0.15)
        # no dearer than the largest listed case
        n = 34.0e6 * 4.0 ** (c["lmax"] - 10) * items / 64 if items else 17.5e6 * 4.0 ** (c["lmax"] - 9)
        slow = (8.0 if c["box"] == 3.0 else 2.5) if c["precision"] == "fp64" else 1.1
        c["iters"] = max(2, min(c["iters"], int(34.0e6 * 50 / (n * slow))))
        return _drop_name(c)
    if u < 0.66:
        return _drop_name(dict(_grid3("", "host", rng.randint(6, 9), log_int(8, 64), iters=rng.randint(5, 20)),
                               precision=rng.choice(["fp64", "mixed"]), order=rng.choice(["2nd", "1st_time"])))
    if u < 0.75:
        lo = rng.randint(5, 8)
        return dict(kind="batch", trees=log_int(48, 512), lmin=3, lmax_lo=lo, lmax_hi=rng.randint(lo, 9),
                    precision=rng.choice(["mixed", "mixed", "fp64"]), iters=rng.randint(10, 20))
    if u < 0.83:
        return _drop_name(_grid3("", "advect", rng.randint(6, 9), log_int(8, 64)))
    if u < 0.91:
        return _drop_name(_grid3("", "curvature", rng.randint(7, 9), log_int(8, 64)))
    if u < 0.95:
        return dict(kind="train", samples=log_int(20000, 131072), batch=rng.choice([4096, 8192, 16384]))
    return _drop_name(dict(_grid3("", "regrid", rng.randint(7, 9), log_int(8, 64), iters=rng.randint(2, 6)),
                           precision=rng.choice(["fp64", "mixed"])))


def _drop_name(c):
    return {k: v for k, v in c.items() if k != "name"}


# ------------------------------------------------------------------ inputs
def _shape(case):
    """The level set that refines a case's grid."""
    box = case["box"]
    if case["shape"] == "star":
        return ls.Star(center=(0.5 * box, 0.5 * box), r0=0.3 * box, amplitude=0.05 * box, lobes=5, k=0.8 / box ** 2)
    if case["shape"] == "gyroid":
        return ls.Gyroid(w=8 * np.pi / box, c=0.3, e=0.5 / box ** 3)
    rng = np.random.default_rng(20261202)
    centers = rng.uniform(0.2, 0.8, size=(case["items"], 3)) * box
    radii = rng.uniform(0.03, 0.08, size=case["items"]) * box
    return ls.Spheres(centers, radii, 0.0 if case["kind"] == "curvature" else 0.5)


def _mirrored(case, seed):
    """The spheres of a regrid case reflected about the box centre along the
    axes that the seed names (another grid of the same size), and the same
    spheres scaled to other slopes for phi0.  Coordinates on a dyadic lattice:
    a reflection is exact."""
    rng = np.random.default_rng(20261202)
    c = np.rint(rng.uniform(0.2, 0.8, size=(case["items"], 3)) * 4096) / 4096
    r = rng.uniform(0.03, 0.08, size=case["items"])
    for a in range(3):
        if (seed >> a) & 1:
            c[:, a] = 1.0 - c[:, a]
    return ls.Spheres(c, r, 0.0), ls.Spheres(c, r, np.random.default_rng(seed).uniform(0.3, 0.6))


def _grid(case, shape):
    dim, box = case["dim"], case["box"]
    return C.DeviceGrid(dim, shape, case["lmin"], case["lmax"], lip=2.4, box_min=[0.0] * dim, box_max=[box] * dim)


def _wave(dim, box, seed):
    """An oblique plane k.x + p: the phase of a smooth wave over the box."""
    rng = np.random.default_rng(seed)
    k = rng.uniform(-1.0, 1.0, size=dim)
    k *= rng.uniform(2.0, 12.0) / np.linalg.norm(k) / box
    return ls.Plane(list(k), rng.uniform(0.0, 2 * np.pi)), rng.uniform(-0.4, 0.4)


def _phi0(case, grid, shape, seed):
    """phi0 at the nodes.  Calls that reinitialize start away from a signed
    distance: the interface shifted by a fraction of a cell, the slopes varied
    over the box.  curvature starts from the distance to the spheres, bent a
    little within and beyond the band |phi| < 1.5h that it samples."""
    plane, shift = _wave(case["dim"], case["box"], seed)
    h = float(grid.dxyz_min().min())
    phi, wave = grid.sample(shape), torch.sin(grid.sample(plane))
    if case["kind"] == "curvature":
        band = 1.5 * h
        return phi + 0.2 * wave * band / math.pi * torch.sin(math.pi / band * phi)
    return (phi + shift * h) * (1.0 + 0.3 * wave)


def _trees(case, seed):
    rng = np.random.default_rng(20261202)
    specs = [(ls.random_star(rng), int(rng.integers(case["lmax_lo"], case["lmax_hi"] + 1)))
             for _ in range(case["trees"])]
    plane, shift = _wave(2, 1.0, seed)

    def one(spec):
        f = C.Forest(2).refine_levelset(spec[0], case["lmin"], spec[1], lip=2.4).build_nodes()
        h = float(np.min(f.dxyz_min()))
        return (C.flat_stencil_from_forest(f),
                (f.sample(spec[0]) + shift * h) * (1.0 + 0.3 * np.sin(f.sample(plane))))

    with ThreadPoolExecutor(8) as ex:
        res = list(ex.map(one, specs))
    return [r[0] for r in res], np.concatenate([r[1] for r in res])


def _velocity(grid, case, seed):
    """A smooth velocity of both signs, about 1 in size."""
    plane, shift = _wave(case["dim"], case["box"], seed + 1)
    return 0.3 * shift + torch.cos(grid.sample(plane))


def _circle_stencils(n, seed):
    """Samples next to circles of radius U[1.6h, 0.5] on an h = 2^-7 grid, as
    curvature.make_dataset takes them from reinitialized level sets: the 3x3
    phi/h stencil and a numerical h*kappa, with the exact h*kappa."""
    h = 2.0 ** -7
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    u = torch.rand((n, 4), dtype=torch.float64, device="cuda", generator=g)
    R = 1.6 * h + (0.5 - 1.6 * h) * u[:, 0]
    th = 2 * math.pi * u[:, 1]
    d = (2 * u[:, 2] - 1) * 0.7 * h  # the node's distance to the circle
    x, y = (R + d) * torch.cos(th), (R + d) * torch.sin(th)
    cols = [(torch.sqrt((x + i * h) ** 2 + (y + j * h) ** 2) - R) / h for i in (-1, 0, 1) for j in (-1, 0, 1)]
    hk = h / R
    cols.append(hk * (1 + 0.2 * (2 * u[:, 3] - 1) * hk))
    return torch.stack(cols, dim=1).float().contiguous(), hk.cpu().numpy()


def prepare(case, seed):
    torch.cuda.init()
    kind, st = case["kind"], {"case": case}
    if kind == "batch":
        tabs, phi0 = _trees(case, seed)
        st["batch"] = C.TreeBatch(tabs)
        st["phi0"] = torch.from_numpy(phi0).cuda()
        st["phi"] = torch.empty_like(st["phi0"])
        st["batch"].autotune(st["phi0"], case["iters"], case["precision"])
        return st
    if kind == "train":
        st["feat"], st["target"] = _circle_stencils(case["samples"], seed)
        st["net"] = CV.CurvatureNet(seed=seed)
        return st
    if kind == "regrid":
        C.device_cache_set_limit(24 << 30)  # as a program that rebuilds its grid in a loop does
        st["shape"], st["shape0"] = _mirrored(case, seed)
        return st
    shape = _shape(case)
    st["grid"] = _grid(case, shape)
    st["grid"].device()
    phi0 = _phi0(case, st["grid"], shape, seed)
    if kind == "host":
        st["phi"] = phi0.cpu().numpy()
    else:
        st["phi0"], st["phi"] = phi0, torch.empty_like(phi0)
    if kind in ("reinit", "host"):
        solver = C.LevelSet(st["grid"], precision=case["precision"], graph=case.get("graph", False))
        st["call"] = getattr(solver, ORDERS[case["order"]][0])
    elif kind == "advect":
        st["solver"] = C.LevelSet(st["grid"])
        st["vn"] = _velocity(st["grid"], case, seed)
    elif kind == "curvature":
        st["net"] = CV.CurvatureNet.load(os.path.join(os.path.dirname(CV.__file__), "weights", "curvature3d.npz"))
        st["h"] = float(st["grid"].dxyz_min().min())
    return st


# ------------------------------------------------------------------ the calls
def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "reinit":
        st["phi"].copy_(st["phi0"])
        return st["call"](st["phi"], case["iters"])
    if kind == "host":
        return st["call"](st["phi"], case["iters"])
    if kind == "batch":
        st["phi"].copy_(st["phi0"])
        return st["batch"].reinitialize_2nd_order(st["phi"], case["iters"], precision=case["precision"])
    if kind == "advect":
        st["phi"].copy_(st["phi0"])
        dt = st["solver"].advect_in_normal_direction(st["vn"], st["phi"])
        return {"phi": st["phi"], "dt": dt}
    if kind == "curvature":
        ds, phi, h = st["grid"].device(), st["phi0"], st["h"]
        nrm = C.compute_normals(st["grid"], phi)
        kap = C.compute_mean_curvature(st["grid"], nrm)
        feat, off, node, skipped = CV.grid_samples(ds, phi, h, 1.5 * h, nrm, kap)
        hk = CV.hybrid_hk(st["net"], feat)
        return {"normals": nrm, "kappa": kap, "feat": feat, "offset": off, "node": node, "skipped": skipped, "hk": hk}
    if kind == "train":
        hist = CV.train(st["net"], st["feat"], st["target"], epochs=1, batch=case["batch"])
        return {"loss": hist["loss"], "params": np.concatenate(st["net"].params())}
    grid = _grid(case, st["shape"])
    phi = grid.sample(st["shape0"])
    C.LevelSet(grid, precision=case["precision"]).reinitialize_2nd_order(phi, case["iters"])
    st["grid"] = grid  # the previous one is dropped
    return {"phi": phi, "sizes": list(grid.sizes())}


# ------------------------------------------------------------------ floors
@functools.lru_cache(maxsize=None)
def _nodes(key):
    """(nodes, leaves) of a nominal grid of the case."""
    case = dict(key)
    if case["kind"] == "batch":
        # one tree's nodes double with each level: about 1300 at level 6
        levels = range(case["lmax_lo"], case["lmax_hi"] + 1)
        return int(case["trees"] * sum(1300 * 2.05 ** (k - 6) for k in levels) / len(levels)), 0
    torch.cuda.init()
    leaves, nodes, _ = _grid(case, _mirrored(case, 0)[0] if case["kind"] == "regrid" else _shape(case)).sizes()
    return nodes, leaves


def work(case):
    """Reinitialization and advection: per stage, read phi, read phi0 or the
    velocity, write phi and one int32 index per face, and (RK2) one more read
    of phi.  Curvature: phi, normals and kappa once, plus the samples.
    Training: the products of the forward and backward passes."""
    if case["kind"] == "train":
        rows = 2 * case["samples"]
        steps = rows // case["batch"]
        dims = CV.DIMS_2D
        macs = sum(i * o for i, o in zip(dims[:-1], dims[1:]))
        return {"bytes": float(4 * rows * (dims[0] + 1) + steps * 4 * 4 * macs),
                "flops": float(2 * steps * case["batch"] * (3 * macs - dims[0] * dims[1]))}
    key = tuple(sorted((k, v) for k, v in case.items() if k != "name"))
    n, leaves = _nodes(key)
    dim = case.get("dim", 2)
    w = 4 if case.get("precision") == "mixed" else 8
    stages = 1 if case.get("order") in ("1st_time", "1st") else 2
    per_iter = stages * (3 * w + 8 * dim) + (w if stages == 2 else 0)
    flops = 20 * dim * stages * case.get("iters", 0) * n
    sweep = per_iter * case.get("iters", 0) * n
    if case["kind"] == "host":
        sweep += 16 * n
    elif case["kind"] == "advect":
        sweep, flops = n * (2 * (24 + 8 * dim) + 8 + 4 * dim), 2 * 20 * dim * n
    elif case["kind"] == "curvature":
        # about a third of the nodes are samples of 28 floats, 3 doubles, an id and a result
        sweep, flops = n * (8 + 2 * 24 + 8 + 8 * dim) + n // 3 * 148, n * 60 + n // 3 * 2 * 53000
    elif case["kind"] == "regrid":
        # leaves, node coordinates, neighbours and distances written once, then the short sweep
        sweep += leaves * 16 + n * (12 + 24 * 4 + 30 * 8 + 8)
    return {"bytes": float(sweep), "flops": float(flops)}


# ------------------------------------------------------------------ 64-bit values
class _Tables:
    """The flattened stencils as torch arrays: corner ids and normalised
    weights per face, arm lengths, and the transverse products d_m0 d_p0."""

    def __init__(self, tabs):
        tabs = tabs if isinstance(tabs, list) else [tabs]
        self.dim = tabs[0].dim
        F, K, D = 2 * self.dim, 2 ** (self.dim - 1), self.dim
        off = np.cumsum([0] + [t.n_nodes for t in tabs])
        self.N, self.zdt = int(off[-1]), tabs[0].zero_distance_threshold

        def cat(get, add=False):
            return torch.cat([torch.from_numpy(get(t)).cuda() + (int(o) if add else 0) for t, o in zip(tabs, off)])

        self.idx = [[cat(lambda t: t.nbr[f, c], True) for c in range(K)] for f in range(F)]
        self.d = [cat(lambda t: t.d[f]) for f in range(F)]
        self.tr = [[cat(lambda t: t.d_tr[f, k]) for k in range(2 * (D - 1))] for f in range(F)]
        wall = cat(lambda t: t.wall)
        self.wall = [(wall & (1 << f)) != 0 for f in range(F)]
        self.P, self.w = [], []
        for f in range(F):
            t = self.tr[f]
            self.P.append([t[2 * k] * t[2 * k + 1] for k in range(D - 1)])
            if D == 2:
                self.w.append([t[1] / (t[0] + t[1]), t[0] / (t[0] + t[1])])
            else:
                nrm = (t[0] + t[1]) * (t[2] + t[3])
                self.w.append([t[1] * t[3] / nrm, t[0] * t[3] / nrm, t[1] * t[2] / nrm, t[0] * t[2] / nrm])
        self.cross_axes = [[b for b in range(D) if b != a] for a in range(D)]
        m = [[torch.ones(self.N, dtype=torch.float64, device="cuda") if a == b else None for b in range(D)]
             for a in range(D)]
        for a in range(D):
            s = self.d[2 * a] + self.d[2 * a + 1]
            for k, b in enumerate(self.cross_axes[a]):
                m[a][b] = self.P[2 * a][k] / self.d[2 * a] / s + self.P[2 * a + 1][k] / self.d[2 * a + 1] / s
        self.inv = _inverse(m)

    def face(self, f, g):
        r = 0.0
        for c, w in enumerate(self.w[f]):
            r = r + w * torch.index_select(g, 0, self.idx[f][c])
        return r

    def second(self, g):
        """(linear face values, second derivatives) of g"""
        fv = [self.face(f, g) for f in range(2 * self.dim)]
        naive = [2 * ((fv[2 * a + 1] - g) / self.d[2 * a + 1] + (fv[2 * a] - g) / self.d[2 * a])
                 / (self.d[2 * a] + self.d[2 * a + 1]) for a in range(self.dim)]
        dd = [sum(self.inv[a][b] * naive[b] for b in range(self.dim)) for a in range(self.dim)]
        return fv, dd

    def quadratic(self, g):
        fv, dd = self.second(g)
        out = []
        for f in range(2 * self.dim):
            v = fv[f]
            for k, b in enumerate(self.cross_axes[f >> 1]):
                v = v - 0.5 * self.P[f][k] * dd[b]
            out.append(v)
        return out, dd

    def gradient(self, g):
        fv, dd = self.second(g)
        out = []
        for a in range(self.dim):
            dm, dp = self.d[2 * a], self.d[2 * a + 1]
            v = ((fv[2 * a + 1] - g) * dm / dp + (g - fv[2 * a]) * dp / dm) / (dp + dm)
            for k, b in enumerate(self.cross_axes[a]):
                v = v - dd[b] * 0.5 * (self.P[2 * a + 1][k] * dm / dp - self.P[2 * a][k] * dp / dm) / (dm + dp)
            out.append(v)
        return out


def _inverse(m):
    """Inverse of a 2x2 or 3x3 matrix of arrays, by cofactors."""
    n = len(m)
    if n == 2:
        det = m[0][0] * m[1][1] - m[0][1] * m[1][0]
        return [[m[1][1] / det, -m[0][1] / det], [-m[1][0] / det, m[0][0] / det]]
    cof = [[m[(i + 1) % 3][(j + 1) % 3] * m[(i + 2) % 3][(j + 2) % 3]
            - m[(i + 1) % 3][(j + 2) % 3] * m[(i + 2) % 3][(j + 1) % 3] for j in range(3)] for i in range(3)]
    det = sum(m[0][j] * cof[0][j] for j in range(3))
    return [[cof[j][i] / det for j in range(3)] for i in range(3)]


def _minmod(a, b):
    return torch.where(a * b <= 0, torch.zeros_like(a), torch.where(a.abs() < b.abs(), a, b))


def _root(a, b, fa, fb, faa, fbb):
    """Zero in (a, b) of the parabola through fa and fb with the smaller second derivative."""
    eps = 1e-13
    fxx = _minmod(faa, fbb)
    h = b - a
    c2, c1, c0 = 0.5 * fxx, (fb - fa) / h, 0.5 * (fb + fa) - h * h / 8 * fxx
    disc = torch.sqrt(torch.clamp(c1 * c1 - 4 * c2 * c0, min=0))
    x = torch.where(c2.abs() < eps, -c0 / c1, -2 * c0 / (c1 + torch.where(fb < 0, -disc, disc))) + 0.5 * (a + b)
    return torch.where(fa.abs() < eps, a + eps, torch.where(fb.abs() < eps, b - eps, x))


def _mirror(T, s, v, dd, ddf):
    """Neumann condition on the walls."""
    for a in range(T.dim):
        for x, y in ((2 * a, 2 * a + 1), (2 * a + 1, 2 * a)):
            w = T.wall[x]
            s[x], v[x] = torch.where(w, s[y], s[x]), torch.where(w, v[y], v[x])
            if ddf is not None:
                z = torch.zeros_like(dd[a])
                dd[a] = torch.where(w, z, dd[a])
                ddf[x], ddf[y] = torch.where(w, z, ddf[x]), torch.where(w, z, ddf[y])


def _one_sided(T, p, s, v, dd, ddf):
    out = []
    for a in range(T.dim):
        dp, dm = (v[2 * a + 1] - p) / s[2 * a + 1], (p - v[2 * a]) / s[2 * a]
        if ddf is not None:
            dm = dm + 0.5 * s[2 * a] * _minmod(ddf[2 * a], dd[a])
            dp = dp - 0.5 * s[2 * a + 1] * _minmod(ddf[2 * a + 1], dd[a])
        out.append((dm, dp))
    return out


def _exact_reinit(T, phi0, space, time, iters):
    F = 2 * T.dim
    anchor, sgn = phi0.abs() < T.zdt, torch.where(phi0 > 0, 1.0, -1.0).double()
    v, dd = T.quadratic(phi0)
    zero = torch.zeros_like(phi0)
    cross, sub = [], []
    for f in range(F):
        a = f >> 1
        cross.append(phi0 * v[f] < 0)
        ddf = T.face(f, dd[a]) if space == 2 else zero
        d0 = dd[a] if space == 2 else zero
        r = -_root(-T.d[f], zero, v[f], phi0, ddf, d0) if f % 2 == 0 else _root(zero, T.d[f], phi0, v[f], d0, ddf)
        sub.append(torch.clamp(r, min=T.zdt))

    def stage(p):
        v, dd = T.quadratic(p)
        ddf = [T.face(f, dd[f >> 1]) for f in range(F)] if space == 2 else None
        s = [torch.where(cross[f], sub[f], T.d[f]) for f in range(F)]
        v = [torch.where(cross[f], zero, v[f]) for f in range(F)]
        _mirror(T, s, v, dd, ddf)
        dt = s[0]
        for f in range(1, F):
            dt = torch.minimum(dt, s[f])
        total = 0.0
        for dm, dp in _one_sided(T, p, s, v, dd, ddf):
            dm, dp = torch.clamp(sgn * dm, min=0), torch.clamp(sgn * dp, max=0)
            total = total + torch.maximum(dm * dm, dp * dp)
        r = p - dt / T.dim * sgn * (torch.sqrt(total) - 1)
        r = torch.where(r * sgn < 0, -r, r)
        return torch.where(anchor, zero, r)

    p = phi0.clone()
    for _ in range(iters):
        q = stage(p)
        p = 0.5 * (p + stage(q)) if time == 2 else q
    return p


def _exact_advect(T, phi, vn):
    s = T.d[0].abs()
    for d in T.d[1:]:
        s = torch.minimum(s, d.abs())
    dt = float((0.8 * (s / vn).abs()).min())

    def stage(p):
        v, dd = T.quadratic(p)
        ddf = [T.face(f, dd[f >> 1]) for f in range(2 * T.dim)]
        s = list(T.d)
        _mirror(T, s, v, dd, ddf)
        sgn = torch.where(vn > 0, 1.0, -1.0).double()
        total = 0.0
        for dm, dp in _one_sided(T, p, s, v, dd, ddf):
            total = total + torch.clamp(sgn * dm, min=0) ** 2 + torch.clamp(sgn * dp, max=0) ** 2
        return p - dt * vn * torch.sqrt(total)

    return {"phi": 0.5 * (phi + stage(stage(phi))), "dt": dt}


def _exact_curvature(T, phi, h, band, net):
    g = T.gradient(phi)
    norm = torch.sqrt(sum(x * x for x in g))
    n = torch.stack([torch.where(norm < 1e-13, torch.zeros_like(norm), x / norm) for x in g])
    kap = sum(T.gradient(n[a])[a] for a in range(3))
    node = torch.nonzero(phi.abs() < band).view(-1)
    total = node.numel()

    def arm(f, at):
        """(the node h away through face f, whether there is one)"""
        ok, corner = T.d[f][at] == h, torch.zeros_like(at)
        for k in range(2):
            low = T.tr[f][2 * k][at] == 0
            ok = ok & (low | (T.tr[f][2 * k + 1][at] == 0))
            corner = corner + torch.where(low, 0, 1 << k)
        ids = torch.stack([T.idx[f][c][at] for c in range(4)])
        return ids.gather(0, corner[None])[0].long(), ok

    blk, good = {(0, 0, 0): node}, torch.ones_like(node, dtype=torch.bool)
    for a in range(3):
        for key in list(blk):
            for side in (0, 1):
                to = list(key)
                to[a] = 2 * side - 1
                blk[tuple(to)], ok = arm(2 * a + side, blk[key])
                good = good & ok
    keep = torch.nonzero(good).view(-1)
    node = node[keep]
    order = [(i, j, k) for i in (-1, 0, 1) for j in (-1, 0, 1) for k in (-1, 0, 1)]
    ids = torch.stack([blk[o][keep] for o in order])
    off = -phi[node] * n[:, node]
    u = torch.clamp(off / h, -1, 1)
    lo = torch.where(u < 0, -1, 0)
    w = u - lo
    ihk = 0.0
    for c in range(8):
        wt, pos = 1.0, 0
        for a in range(3):
            bit = (c >> a) & 1
            wt = wt * (w[a] if bit else 1 - w[a])
            pos = pos * 3 + (lo[a] + bit + 1)
        ihk = ihk + wt * kap[ids.gather(0, pos[None])[0]]
    feat = torch.cat([phi[ids] / h, (h * ihk)[None]]).T.contiguous()
    return {"normals": n, "kappa": kap, "feat": feat, "offset": off.T.contiguous(), "node": node,
            "skipped": total - node.numel(), "hk": _exact_learned(feat, net)}


def _mlp(x, dims, w, b):
    o = ob = 0
    for l, (i, k) in enumerate(zip(dims[:-1], dims[1:])):
        x = x @ w[o:o + i * k].view(i, k) + b[ob:ob + k]
        o, ob = o + i * k, ob + k
        if l < len(dims) - 2:
            x = torch.relu(x)
    return x


def _double(x):
    return torch.as_tensor(np.asarray(x), dtype=torch.float64, device="cuda")


def _exact_learned(feat, net):
    """The hybrid h*kappa of 3x3x3 samples: one orientation of the cube, the
    plane-deviation basis, the network, the blend."""
    lo, hi = CV.LO_MIN_HK, CV.UP_MIN_HK
    w, b = (_double(x) for x in net.params())
    mean, std = _double(net.mean), _double(net.std)
    out = []
    for f in torch.split(feat, 1 << 20):
        ihk = f[:, 27]
        f = torch.where(ihk > 0, -1.0, 1.0).double()[:, None] * f
        v = f[:, :27].reshape(-1, 3, 3, 3)
        rows = torch.arange(v.shape[0], device=v.device)
        g = torch.stack([v[:, 2, 1, 1] - v[:, 0, 1, 1], v[:, 1, 2, 1] - v[:, 1, 0, 1],
                         v[:, 1, 1, 2] - v[:, 1, 1, 0]], dim=1)
        p = torch.sort(g.abs(), dim=1, descending=True, stable=True).indices
        r = torch.where(g < 0, -1, 1)
        grid = torch.empty_like(v)
        for i in (-1, 0, 1):
            for j in (-1, 0, 1):
                for k in (-1, 0, 1):
                    c = torch.zeros_like(p)
                    for axis, o in enumerate((i, j, k)):
                        c.scatter_(1, p[:, axis:axis + 1], o * r.gather(1, p[:, axis:axis + 1]))
                    grid[:, i + 1, j + 1, k + 1] = v[rows, c[:, 0] + 1, c[:, 1] + 1, c[:, 2] + 1]
        v = grid
        f0 = v[:, 1, 1, 1]
        gx, gy, gz = (0.5 * (a - c) for a, c in ((v[:, 2, 1, 1], v[:, 0, 1, 1]), (v[:, 1, 2, 1], v[:, 1, 0, 1]),
                                                 (v[:, 1, 1, 2], v[:, 1, 1, 0])))
        o = torch.tensor([-1.0, 0.0, 1.0], dtype=torch.float64, device=v.device)
        plane = (f0[:, None, None, None] + gx[:, None, None, None] * o.view(1, 3, 1, 1)
                 + gy[:, None, None, None] * o.view(1, 1, 3, 1) + gz[:, None, None, None] * o.view(1, 1, 1, 3))
        x = v - plane
        x[:, 1, 1, 1], x[:, 0, 1, 1], x[:, 1, 0, 1], x[:, 1, 1, 0] = f0, gx, gy, gz
        x = torch.cat([x.reshape(-1, 27), f[:, 27:]], dim=1)
        pred = _mlp((x - mean) / std, net.dims, w, b)[:, 0]
        a = ihk.abs()
        q = torch.where(pred.abs() > net.deadband, pred, torch.zeros_like(pred)) - a
        lam = (hi - a) / (hi - lo)
        q = torch.where(a <= hi, (1 - lam) * q - lam * a, q)
        out.append(torch.where(a < lo, ihk, torch.where(ihk > 0, q.abs(), -q.abs())))
    return torch.cat(out)


def _exact_train(st):
    """curvature.train's epoch in 64 bits: the same batches, Adam, and the
    output scale folded into the last layer."""
    case, net = st["case"], st["net"]
    f, t = st["feat"].double(), _double(st["target"])
    ihk = f[:, 9]
    s = torch.where(ihk > 0, -1.0, 1.0).double()
    v = (s[:, None] * f)[:, :9].reshape(-1, 3, 3)
    gx, gy = v[:, 2, 1] - v[:, 0, 1], v[:, 1, 2] - v[:, 1, 0]
    quad = torch.where(gy < 0, torch.where(gx < 0, 2, 3), torch.where(gx < 0, 1, 0))
    rot = v.clone()
    for k, turns in ((1, -1), (2, 2), (3, 1)):
        rot[quad == k] = torch.rot90(v[quad == k], turns, dims=(1, 2))
    one = torch.cat([rot.reshape(-1, 9), (s * ihk)[:, None]], dim=1)
    two = torch.cat([rot.transpose(1, 2).reshape(-1, 9), (s * ihk)[:, None]], dim=1)
    x = torch.stack([one, two], dim=1).reshape(-1, 10)
    y = (s * t + ihk.abs()).repeat_interleave(2)
    x = (x - x.mean(dim=0)) / x.std(dim=0).clamp_min(1e-6)
    sigma = float(y.std().clamp_min(1e-12))
    y = y / sigma
    w, b = (_double(p).requires_grad_() for p in net.params())
    n, batch = x.shape[0], case["batch"]
    steps = max(1, n // batch)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(0)
    perm = torch.randperm(n, device="cuda", generator=gen)
    opt = torch.optim.Adam([w, b], lr=1e-3, betas=(0.9, 0.999), eps=1e-8)
    loss_sum = 0.0
    for k in range(steps):
        at = perm[k * batch:(k + 1) * batch]
        opt.param_groups[0]["lr"] = 1e-5 + 0.5 * (1e-3 - 1e-5) * (1 + math.cos(math.pi * k / max(1, steps - 1)))
        opt.zero_grad()
        loss = ((_mlp(x[at], net.dims, w, b)[:, 0] - y[at]) ** 2).mean()
        loss.backward()
        opt.step()
        loss_sum += float(loss.detach())
    w, b = w.detach().clone(), b.detach().clone()
    w[-net.dims[-2]:] *= sigma
    b[-1:] *= sigma
    return {"loss": [loss_sum / steps], "params": torch.cat([w, b])}


def exact(case, seed):
    kind = case["kind"]
    if kind == "train":
        return _exact_train(prepare(case, seed))
    if kind == "batch":
        tabs, phi0 = _trees(case, seed)
        return _exact_reinit(_Tables(tabs), torch.from_numpy(phi0).cuda(), 2, 2, case["iters"])
    shape, shape0 = _mirrored(case, seed) if kind == "regrid" else (_shape(case), None)
    grid = _grid(case, shape)
    phi = grid.sample(shape0) if kind == "regrid" else _phi0(case, grid, shape, seed)
    _, space, time = ORDERS[case.get("order", "2nd")]
    if kind in ("reinit", "host", "regrid") and phi.numel() * case["iters"] * time > 6.0e8:
        return None  # over about 20 seconds
    T = _Tables(grid.tables())
    if kind in ("reinit", "host"):
        return _exact_reinit(T, phi, space, time, case["iters"])
    if kind == "advect":
        return _exact_advect(T, phi, _velocity(grid, case, seed))
    if kind == "curvature":
        h = float(grid.dxyz_min().min())
        net = CV.CurvatureNet.load(os.path.join(os.path.dirname(CV.__file__), "weights", "curvature3d.npz"))
        return _exact_curvature(T, phi, h, 1.5 * h, net)
    return {"phi": _exact_reinit(T, phi, 2, 2, case["iters"]), "sizes": list(grid.sizes())}
